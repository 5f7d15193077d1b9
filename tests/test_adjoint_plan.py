"""Which slices the adjoint takes together (adj_groups in
acumen_amd/csrc/grad.hip), checked on the CPU through the built library: every
slice is in one group, of its geometry and of at most the size asked for, with
at most one group of a geometry not full, a slice without a partner is a group
of its own, and groups of longer tiles come first."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "acumen_amd")

CHECKER = r"""
#include <algorithm>
#include <cstdio>
#include <map>
#include <random>
#include <vector>
namespace acu {
std::vector<std::vector<int>> adj_groups(const std::vector<int>& geo, const std::vector<int>& T, int most);
}
static int width(size_t n) { return n <= 2 ? (int)n : n <= 4 ? 4 : 8; }
static int check_groups(const std::vector<int>& geo, const std::vector<int>& T, int most) {
  const auto g = acu::adj_groups(geo, T, most);
  std::vector<int> seen(geo.size(), 0);
  std::map<int, std::vector<int>> sizes;
  for (size_t i = 0; i < g.size(); ++i) {
    if (g[i].empty() || (int)g[i].size() > most) return 1;
    // neither more angles nor more slices than every group before it
    for (size_t j = 0; j < i; ++j)
      if (T[g[i][0]] >= T[g[j][0]] && width(g[i].size()) >= width(g[j].size()) &&
          T[g[i][0]] * width(g[i].size()) > T[g[j][0]] * width(g[j].size())) return 2;
    for (int v : g[i]) {
      if (v < 0 || v >= (int)geo.size() || seen[v]++ || geo[v] != geo[g[i][0]]) return 3;
    }
    sizes[geo[g[i][0]]].push_back((int)g[i].size());
  }
  for (int v : seen) if (!v) return 4;
  for (auto& p : sizes) {  // full groups and at most one remainder
    const int n = (int)std::count(geo.begin(), geo.end(), p.first);
    if ((int)p.second.size() != (n + most - 1) / most) return 5;
    std::sort(p.second.begin(), p.second.end());
    for (size_t i = 1; i < p.second.size(); ++i) if (p.second[i] != most) return 6;
  }
  return 0;
}
int main() {
  std::mt19937 rng(5);
  for (int it = 0; it < 300; ++it) {
    const int n = 1 + rng() % 40, kinds = 1 + rng() % 8;
    std::vector<int> geo(n), T(n), Tk(kinds);
    for (auto& v : Tk) v = 1 + rng() % 1500;
    for (int i = 0; i < n; ++i) T[i] = Tk[geo[i] = rng() % kinds];
    for (int most : {1, 2, 4, 8})
      if (int e = check_groups(geo, T, most)) { std::printf("groups %d\n", e); return 1; }
  }
  // five of one geometry among single slices; nine of one
  std::vector<int> geo = {0, 1, 0, 2, 0, 3, 0, 4, 0};
  auto g = acu::adj_groups(geo, std::vector<int>(9, 60), 8);
  if (g.size() != 5 || g[0].size() != 5 || g[1].size() != 1) { std::printf("mixed\n"); return 1; }
  g = acu::adj_groups(std::vector<int>(9, 0), std::vector<int>(9, 60), 8);
  if (g.size() != 2 || g[0].size() != 8 || g[1].size() != 1) { std::printf("nine\n"); return 1; }
  std::printf("ok\n");
  return 0;
}
"""


def test_groups(tmp_path):
    if not os.path.exists(os.path.join(LIB, "libacumen_hip.so")):
        pytest.fail("libacumen_hip.so not built (python -c 'import __graft_entry__ as g; g.build()')")
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(CHECKER)
    subprocess.run([cxx, "-O1", "-std=c++17", str(src), "-L", LIB, "-lacumen_hip", f"-Wl,-rpath,{LIB}", "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
