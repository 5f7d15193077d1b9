"""The median of three sorted rows (acumen_amd/csrc/median_net.hpp: sort9 and
median27_of_sorted, used by the preprocessing median filter,
projections_to_sinogram_hpc.F90:420-447), checked on all 2^27 binary inputs:
min3, med3 and max3 are threshold functions, so by the 0-1 principle what
selects the median of every 0-1 input selects it of every totally ordered
input."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "acumen_amd", "csrc")

PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include "median_net.hpp"
typedef uint64_t V;  // 64 binary inputs side by side
struct Bits {
  static V min3(V a, V b, V c) { return a & b & c; }
  static V med3(V a, V b, V c) { return (a & b) | (a & c) | (b & c); }
  static V max3(V a, V b, V c) { return a | b | c; }
};
int main() {
  static const V pat[6] = {0xAAAAAAAAAAAAAAAAull, 0xCCCCCCCCCCCCCCCCull, 0xF0F0F0F0F0F0F0F0ull,
                           0xFF00FF00FF00FF00ull, 0xFFFF0000FFFF0000ull, 0xFFFFFFFF00000000ull};
  long bad = 0;
  for (V w = 0; w < (V)1 << 21; ++w) {
    V in[27], v[3][9];
    for (int j = 0; j < 27; ++j) in[j] = j < 6 ? pat[j] : ((w >> (j - 6)) & 1 ? ~(V)0 : 0);
    V want = 0;
    for (int l = 0; l < 64; ++l)
      if (__builtin_popcountll(w) + __builtin_popcount((unsigned)l) >= 14) want |= (V)1 << l;
    for (int j = 0; j < 27; ++j) v[j / 9][j % 9] = in[j];
    for (auto& r : v) {
      acu::sort9<Bits>(r);
      for (int i = 0; i < 8; ++i) bad += (r[i] & ~r[i + 1]) != 0;
    }
    bad += acu::median27_of_sorted<Bits>(v[0], v[1], v[2]) != want;
  }
  std::printf("%ld\n", bad);
}
"""


def test_selects_the_median_of_every_binary_input(tmp_path):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.strip() == "0"
