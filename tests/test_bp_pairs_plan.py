"""When the backprojector takes slices in pairs (bp_use_pairs) and how much LDS a
launch asks for so that it spreads evenly (bp_pad, both in
acumen_amd/csrc/bp.hip), checked on the CPU through the built library."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "acumen_amd")

CHECKER = r"""
#include <cstdio>
#include <initializer_list>
namespace acu { bool bp_use_pairs(int tiles, int paired); int bp_pad(int active, int own); }
int main() {
  // a launch's few pairs among single slices, and launches of few tiles, stay single
  if (acu::bp_use_pairs(25582, 40) || acu::bp_use_pairs(9162, 816) || acu::bp_use_pairs(1360, 1360)) return 1;
  if (acu::bp_use_pairs(3456, 3456) || acu::bp_use_pairs(6534, 5940) || acu::bp_use_pairs(8840, 0) || acu::bp_use_pairs(0, 0))
    return 2;
  if (!acu::bp_use_pairs(68112, 68112) || !acu::bp_use_pairs(25542, 17028) || !acu::bp_use_pairs(5096, 5096)) return 3;
  if (!acu::bp_use_pairs(2147483646, 2147483646)) return 4;
  // max(3, ceil(share / 32)) workgroups fit a CU of 160 KiB and one more does
  // not, where the kernel's own LDS has room for more; at most 64 KiB in all
  for (int own : {18720, 21776, 25088, 33280}) {
    if (acu::bp_pad(0, own) != 0) return 5;
    for (int share : {1, 32, 33, 70, 96, 97, 128, 129, 160, 161, 192, 193, 500, 268435424}) {
      const int pad = acu::bp_pad(share, own), total = own + pad;
      if (pad < 0 || total > 65536) return 6;
      const int k = share <= 96 ? 3 : (share + 31) / 32;
      const int fit = 163840 / ((total + 1279) / 1280 * 1280), room = 163840 / own;
      if (fit != (room > k ? k : room)) { std::printf("%d %d: %d\n", own, share, fit); return 7; }
    }
  }
  std::printf("ok\n");
  return 0;
}
"""


def test_pairs_rule_and_pad(tmp_path):
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
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stdout + r.stderr)
