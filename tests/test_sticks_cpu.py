"""The host tables of the sphere-pruned transforms: every index that the plane passes take from them lies in the
image that they fill, and the two directions agree. Compiled for the CPU from the library's own header."""
import os
import subprocess

import pytest

from conftest import ROOT

MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include "sticks.hpp"
using namespace pwk;
#define CHECK(x) do { if (!(x)) { std::printf("failed: %s (line %d)\n", #x, __LINE__); return 1; } } while (0)
int main(int argc, char** argv) {
  const int dims[3] = {atoi(argv[1]), atoi(argv[2]), atoi(argv[3])}, r = atoi(argv[4]), shift = atoi(argv[5]);
  std::vector<int32_t> m;
  for (int a = -r; a <= r; ++a)
    for (int b = -r; b <= r; ++b)
      for (int c = -r; c <= r; ++c)
        if (a * a + b * b + c * c <= r * r) { m.push_back(a + shift); m.push_back(b); m.push_back(c); }
  const char* why = nullptr;
  const StickTables t = stick_tables(dims, (int)m.size() / 3, m.data(), &why);
  CHECK(!why);
  const int nx = dims[0], ny = dims[1], S = (int)t.pw0.size(), nx1 = (int)t.x1list.size(), ld = ny + 1;
  CHECK((int)t.st_off.size() == S && (int)t.cnt.size() == S && (int)t.lo.size() == S);
  int waves = 0;
  for (int s = 0; s < S; ++s) { CHECK(t.pw0[s] == waves); waves += t.cnt[s]; }
  CHECK(waves == (int)m.size() / 3);
  for (int32_t g : t.g2fft) CHECK(g >= 0 && g < nx * ny * dims[2]);
  // general image: pl_rows rows filled; the x-lines read rows 0..nx1 (nx1 the zero row) and write up to row
  // nx1 + 1 when the columns are two runs, else rows 0..nx-1
  CHECK((int)t.pl_src.size() == t.pl_rows * ld);
  CHECK(t.x1_runs ? t.pl_rows == nx1 + 1 && t.pl_ra + t.pl_rb == nx1 : t.pl_rows == nx && t.pl_ra == nx && t.pl_rb == 0);
  int used = 0;
  for (int e = 0; e < (int)t.pl_src.size(); ++e)
    if (t.pl_src[e] >= 0) { CHECK(t.pl_src[e] < S && t.st_off[t.pl_src[e]] == e && e % ld < ny); ++used; }
  CHECK(used == S);
  for (int s = 0; s < S; ++s) {
    CHECK(t.st_off[s] >= 0 && t.st_off[s] < t.pl_rows * ld);
    const int row = t.st_off[s] / ld, i1 = t.g2fft[t.pw0[s]] / (ny * dims[2]);
    const int want = i1 < t.pl_ra ? i1 : i1 >= nx - t.pl_rb ? i1 - (nx - t.pl_rb) + t.pl_ra : -1;  // plane_row()
    CHECK(row == want);
  }
  if (t.quarter) {
    const int px = (nx - 1) / 4, py = (ny - 1) / 4, rx = 2 * px + 1, ry = 2 * py + 1, qld = ny | 1;
    CHECK((int)t.q_src.size() == rx * ry && (int)t.q_off.size() == S);
    used = 0;
    for (int e = 0; e < rx * ry; ++e)
      if (t.q_src[e] >= 0) {
        const int s = t.q_src[e], col = e % ry, index = col < py + 1 ? col : col + (ny - ry);  // Quarter::index()
        CHECK(s < S && t.q_off[s] == e / ry * qld + index);
        ++used;
      }
    CHECK(used == S);
    for (int s = 0; s < S; ++s) CHECK(t.q_off[s] >= 0 && t.q_off[s] < rx * qld && t.q_off[s] % qld < ny);
    for (int s = 0; s < S; ++s) CHECK(t.cnt[s] <= 2 * ((dims[2] - 1) / 4) + 1);
  }
  std::printf("%d %d\n", (int)t.quarter, (int)t.x1_runs);
  return 0;
}
"""


@pytest.fixture(scope="module")
def tables(tmp_path_factory):
    d = tmp_path_factory.mktemp("sticks")
    (d / "main.cpp").write_text(MAIN)
    csrc = os.path.join(ROOT, "pwdft-rs_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-D_GLIBCXX_ASSERTIONS", "-I", csrc,
                    str(d / "main.cpp"), "-o", str(d / "tables")], check=True)
    return str(d / "tables")


# (grid, radius, shift of n1): within a quarter of the axes and beyond, every row and all but one, one plane wave,
# unequal axes, the 81-point grids, columns that are not two runs
@pytest.mark.parametrize("dims,m,shift,quarter,runs", [
    ((15, 15, 18), 7, 0, 0, 0), ((16, 16, 16), 7, 0, 0, 1), ((16, 16, 12), 2, 0, 1, 1), ((25, 25, 25), 6, 0, 1, 1),
    ((25, 25, 25), 7, 0, 0, 1), ((8, 8, 8), 0, 0, 1, 1), ((50, 25, 25), 6, 0, 1, 1), ((25, 50, 27), 6, 0, 1, 1),
    ((60, 60, 60), 14, 0, 1, 1), ((64, 32, 30), 7, 0, 1, 1), ((81, 81, 72), 3, 0, 1, 1), ((81, 81, 81), 20, 0, 1, 1),
    ((81, 81, 72), 30, 0, 0, 1), ((81, 81, 72), 17, 0, 1, 1), ((90, 96, 100), 11, 0, 0, 1), ((27, 27, 27), 3, 9, 0, 0)])
def test_every_index_lies_in_its_image(tables, dims, m, shift, quarter, runs):
    out = subprocess.run([tables, *map(str, dims), str(m), str(shift)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    assert out.stdout.split() == [str(quarter), str(runs)]
