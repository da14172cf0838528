// Host side of the sphere-pruned transforms: the z-sticks of a basis and where they lie in the LDS images of a
// z-plane (planes.hpp, Context). No device code, so that every index can be checked without a GPU.
#pragma once

#include <cstdint>
#include <cstdlib>
#include <map>
#include <vector>

#include "fft_sizes.hpp"

namespace pwk {

struct StickTables {
  std::vector<int32_t> g2fft;         // flat grid index of each plane wave
  std::vector<int32_t> pw0, cnt, lo;  // per stick: first plane wave, how many, n3 of the first
  std::vector<int32_t> x1list;        // distinct wrapped i1 that carry sticks, ascending
  bool x1_runs = false;               // they are [0, x1_ra) and [nx - x1_rb, nx): a sphere's columns
  int x1_ra = 0, x1_rb = 0;
  // general image, rows of ny + 1: the rows held (a zero row last when x1_runs) and the runs as the plane
  // passes index them, the stick of each element (-1: zero) and the element of each stick
  int pl_rows = 0, pl_ra = 0, pl_rb = 0;
  std::vector<int32_t> pl_src, st_off;
  // every index within a quarter of its axis (planes.hpp, Quarter): the stick of each held (row, column), and
  // the element of each stick in an image with rows of ny | 1
  bool quarter = false;
  std::vector<int32_t> q_src, q_off;
};

inline int wrap_index(int n, int d) { return ((n % d) + d) % d; }

// m: npw Miller indices in the reference's n1 -> n2 -> n3 order (src/basis.rs:47-59). *why is set when the
// basis has no such tables.
inline StickTables stick_tables(const int dims[3], int npw, const int32_t* m, const char** why) {
  const int nx = dims[0], ny = dims[1], nz = dims[2];
  StickTables t;
  t.g2fft.resize((size_t)npw);
  std::vector<int32_t> xy;
  std::map<int, int> x1index, seen;
  for (int i = 0; i < npw; ++i) {
    const int n1 = m[3 * i], n2 = m[3 * i + 1], n3 = m[3 * i + 2];
    const int col = wrap_index(n1, nx) * ny + wrap_index(n2, ny);
    t.g2fft[(size_t)i] = (int32_t)((size_t)col * nz + wrap_index(n3, nz));
    const bool cont = i > 0 && m[3 * i - 3] == n1 && m[3 * i - 2] == n2 && m[3 * i - 1] + 1 == n3;
    if (!cont) {
      if (!seen.emplace(col, 0).second) {
        *why = "basis is not ordered n1 -> n2 -> n3 or two sticks alias on the grid";
        return t;
      }
      t.pw0.push_back(i);
      t.cnt.push_back(0);
      t.lo.push_back(n3);
      xy.push_back(col);
      x1index[col / ny] = 0;
    }
    if (++t.cnt.back() > nz) {
      *why = "a z-stick is longer than nz (basis aliases on the grid)";
      return t;
    }
  }
  for (auto& kv : x1index) {
    kv.second = (int)t.x1list.size();
    t.x1list.push_back(kv.first);
  }
  const int nx1 = (int)t.x1list.size();
  int ra = 0;
  while (ra < nx1 && t.x1list[(size_t)ra] == ra) ++ra;
  const int rb = nx1 - ra;
  t.x1_runs = nx1 < nx;
  for (int r = 0; r < rb && t.x1_runs; ++r) t.x1_runs = t.x1list[(size_t)(ra + r)] == nx - rb + r;
  t.x1_ra = t.x1_runs ? ra : 0;
  t.x1_rb = t.x1_runs ? rb : 0;
  const int ld = ny + 1;
  t.pl_rows = t.x1_runs ? nx1 + 1 : nx;
  t.pl_ra = t.x1_runs ? ra : nx;
  t.pl_rb = t.x1_runs ? rb : 0;
  t.pl_src.assign((size_t)t.pl_rows * ld, -1);
  for (size_t s = 0; s < xy.size(); ++s) {
    const int i1 = xy[s] / ny;
    t.st_off.push_back((t.x1_runs ? x1index[i1] : i1) * ld + xy[s] % ny);
    t.pl_src[(size_t)t.st_off.back()] = (int32_t)s;
  }
  t.quarter = fft_len_compiled(nx) && fft_len_compiled(ny) && fft_len_compiled(nz);
  for (int i = 0; i < npw && t.quarter; ++i)
    for (int d = 0; d < 3; ++d) t.quarter = t.quarter && std::abs(m[3 * i + d]) <= (dims[d] - 1) / 4;
  if (t.quarter) {
    const int px = (nx - 1) / 4, py = (ny - 1) / 4, rx = 2 * px + 1, ry = 2 * py + 1, qld = ny | 1;
    t.q_src.assign((size_t)rx * ry, -1);
    for (size_t s = 0; s < xy.size(); ++s) {
      const int i1 = xy[s] / ny, i2 = xy[s] % ny;
      const int h1 = i1 <= px ? i1 : i1 - (nx - rx), h2 = i2 <= py ? i2 : i2 - (ny - ry);
      t.q_src[(size_t)h1 * ry + h2] = (int32_t)s;
      t.q_off.push_back(h1 * qld + i2);
    }
  }
  return t;
}

}  // namespace pwk
