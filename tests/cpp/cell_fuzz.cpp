// visit_cell and tile_window (stampcore.hpp) against the window walk they
// stand for, on the CPU: for random imprint geometries and cell boxes, every
// window offset that falls on a cell of the box gets the same cell and pixel
// and lies in the tile window, and the neighbour it names is exactly the other
// visitor of its cell -- any angle (multiples of 45 and 90 degrees among them),
// whole, half and fractional centres, stamps across every canvas edge.  And
// tile_row against the division, for every tile of up to 725 x 725, and Divisor
// (internal.hpp) around the multiples of every kind of divisor.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <utility>
#include <vector>

#include "handles.hpp"
#include "internal.hpp"
#include "stampcore.hpp"

using namespace pnt;

// The reference's index math (FootprintBrush.hxx:90-113) as written there,
// with std::round: stamp_visit must give the same.
static int walk_visit(const StampGeom& g, int col, int row, const FpBox& b, int64_t* ic) {
#pragma clang fp contract(off)
  if (col < -g.hr || col > g.hr || row < -g.hr || row > g.hr) return -1;
  const int x = (int)(col + g.cx), y = (int)(row + g.cy);
  if (y < 0 || x < 0 || x >= g.cols || y >= g.rows) return -1;
  const double rc = col * g.c - row * g.s, rr = col * g.s + row * g.c;
  const int mx = (int)std::round(rc + (double)g.hr), my = (int)std::round(rr + (double)g.hr);
  if (my < 0 || mx < 0 || mx >= g.size_map || my >= g.size_map) return -1;
  if (mx < b.x0 || mx > b.x1 || my < b.y0 || my > b.y1) return -1;
  *ic = (int64_t)y * g.cols + x;
  return my * g.size_map + mx;
}

int main(int argc, char** argv) {
  const int cases = argc > 1 ? std::atoi(argv[1]) : 2000;
  std::mt19937_64 rng(20240607);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  const double kPi = 3.141592653589793238462643383279502884;
  long fail = 0, cells = 0, pairs = 0;
  for (int it = 0; it < cases; ++it) {
    StampGeom g;
    g.size_map = 1 + (int)(U(rng) * (it % 50 == 0 ? 400 : 60));
    g.hr = (g.size_map - 1) / 2;
    g.rows = 1 + (int)(U(rng) * 120);
    g.cols = 1 + (int)(U(rng) * 120);
    const int kind = it % 4;
    g.cx = (U(rng) * 1.4 - 0.2) * g.cols;
    g.cy = (U(rng) * 1.4 - 0.2) * g.rows;
    if (kind == 1) g.cx = std::floor(g.cx), g.cy = std::floor(g.cy);
    if (kind == 2) g.cx = std::floor(g.cx) + 0.5, g.cy = std::floor(g.cy) - 0.5;
    double theta = (U(rng) * 4.0 - 2.0) * kPi;
    if (it % 5 == 0) theta = 0.25 * kPi * std::floor(U(rng) * 17.0 - 8.0);
    if (it % 5 == 1) theta = std::atan2(std::floor(U(rng) * 9.0 - 4.0), std::floor(U(rng) * 9.0 - 4.0));
    g.c = std::cos(-theta);
    g.s = std::sin(-theta);
    FpBox box{0, 0, g.size_map - 1, g.size_map - 1};
    if (it % 3) {
      const int pad = (int)(U(rng) * 0.3 * g.size_map);
      box = FpBox{pad, pad, g.size_map - 1 - pad - (it % 7 == 0), g.size_map - 1 - pad};
    }
    const int side = 2 * g.hr + 1;
    std::vector<std::vector<std::pair<int, int>>> want((size_t)g.size_map * g.size_map);
    for (int row = -g.hr; row <= g.hr; ++row)
      for (int col = -g.hr; col <= g.hr; ++col) {
        int64_t ic;
        const int m = walk_visit(g, col, row, box, &ic);
        if (m >= 0) want[(size_t)m].push_back({col, row});
      }
    const TileWin w = tile_window(g, box);
    long seen = 0, visits = 0;
    for (auto& v : want) visits += (long)v.size();
    for (int row = -g.hr - 2; row <= g.hr + 2; ++row)
      for (int col = -g.hr - 2; col <= g.hr + 2; ++col) {
        int64_t ic = -1;
        const int m = walk_visit(g, col, row, box, &ic);
        const VisitCell V = visit_cell(g, box, col, row);
        int64_t i2 = -1;
        const FpBox all{0, 0, g.size_map - 1, g.size_map - 1};
        bool ok = V.mm == m && stamp_visit(g, col, row, &i2) == walk_visit(g, col, row, all, &ic) &&
                  (m < 0 || i2 == ic);
        if (ok && m >= 0) {
          const auto& c = want[(size_t)m];
          ok = (int64_t)V.y * g.cols + V.x == ic && c.size() <= 2 &&
               col >= w.col0 && col < w.col0 + w.cols && row >= w.row0 && row < w.row0 + w.rows;
          static const int dx[5] = {0, -1, 0, 1, 0}, dy[5] = {0, 0, -1, 0, 1};
          const bool first = c[0] == std::make_pair(col, row);
          if (c.size() == 1) ok = ok && V.shared == 0;
          if (c.size() == 2)
            ok = ok && c[first ? 1 : 0] == std::make_pair(col + dx[V.shared], row + dy[V.shared]) &&
                 (V.shared >= 3) == first;
          ++seen;
          pairs += c.size() == 2 && first;
        }
        ++cells;
        if (!ok && fail++ < 10)
          std::fprintf(stderr, "case %d: offset (%d, %d) of %d: cell %d (want %d), shared %d\n", it,
                       col, row, side, V.mm, m, V.shared);
      }
    if (seen != visits) ++fail;
  }
  // the rows' first and last tiles: tile_row rises with the tile; the
  // hardware's reciprocal is within an ulp
  for (int tx = 1; tx <= 725; ++tx) {
    const float r0 = 1.0f / (float)tx;
    for (const float r : {std::nextafter(r0, 0.0f), r0, std::nextafter(r0, 2.0f)})
      for (int ty = 0; ty < 725; ++ty)
        if (tile_row(ty * tx, r) != ty || tile_row(ty * tx + tx - 1, r) != ty) ++fail;
  }
  for (int it = 0; it < 20000; ++it) {
    const uint32_t d = it < 3000 ? 1u + (uint32_t)it : 1u + (uint32_t)(rng() >> (1 + rng() % 31 + 32));
    const Divisor D = Divisor::of(d);
    for (int k = 0; k < 64; ++k) {
      const uint32_t n = k < 4 ? 0xffffffffu - (uint32_t)k : (uint32_t)(rng() >> (32 + rng() % 31));
      for (const uint32_t v : {n, n / d * d, n / d * d - 1u, n / d * d + d - 1u})
        if (D.div(v) != v / d) ++fail;
    }
  }
  std::printf("%d stamps, %ld offsets, %ld shared cells: %ld failures\n", cases, cells,
              pairs, fail);
  return fail || !pairs ? 1 : 0;
}
