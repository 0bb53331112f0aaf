// How the direct coupling transform cuts its work, by size and precision.  Plain
// C++: no device code.
#pragma once

#include <algorithm>
#include <cstddef>

namespace phx {

// Workgroups of `rows` inner points, 4 / wc waves of mt 16-row tiles by wc waves
// of nt 16-column tiles, the panel columns in windows of `modes` whole modes.
struct CoupTiling {
  int mt, nt, wc, rows, modes;
  int stage;   // the g3 tile's LDS holds the rows' frequencies and energies once g3 has been used
  size_t lds;  // beyond 160 KB: the sizes are not supported
};

constexpr size_t kCoupReduceLds = 1024;  // of reduce_partials

// As few windows as fit: whole panels of up to 24 column tiles (FP32) or 12
// (FP64, whose tiles take twice the registers and LDS), and fewer modes per window
// where g' and |g|^2 of a row tile leave less LDS to g3.  One column wave up to 3
// tiles, two up to 8, four beyond; the other waves take rows.  Several windows
// leave a row tile's g' in LDS between them, so they run 16 rows per workgroup.
// Four column waves take two row tiles each, which serve both from one load of the
// panel, when more than 256 workgroups of 32 points do not fit the card at once as
// twice as many of 16 points do.  18 modes x 16 bands in FP32, us per launch with
// 32 and 16 points: 108 workgroups of 32 points 81 and 55, 256 83 and 64, 432 114
// and 120, 3348 644 and 730; 12 x 16 in FP64 64 and 40, 67 and 52, 91 and 93, 513
// and 542.
inline CoupTiling coupling_tiling(bool f64, int nm, int nw, int nb2max, int points, int nPanels) {
  auto ceil = [](int a, int b) { return (a + b - 1) / b; };
  CoupTiling c{};
  const size_t scratch = size_t(16) * nm * nb2max * (16 + 8);
  const int most = f64 ? 192 : 384;
  int windows = ceil(nm, std::max(1, most / nw));
  c.modes = ceil(nm, windows);
  for (;;) {
    windows = ceil(nm, c.modes);
    const size_t g3 = (size_t(16) * c.modes * nw * (f64 ? 16 : 8) + 15) / 16 * 16;
    c.stage = g3 >= size_t(16) * (nm + nb2max) * 8;
    c.lds = std::max(g3 + scratch, kCoupReduceLds);
    if (c.lds <= 160 * 1024 || c.modes == 1) break;
    // even windows, and at least one mode less: ceil(nm / (windows + 1)) can be the same number of modes
    c.modes = std::min(c.modes - 1, ceil(nm, windows + 1));
  }
  const int tiles = ceil(c.modes * nw, 16);
  c.wc = windows > 1 ? 4 : tiles <= 3 ? 1 : tiles <= 8 ? 2 : 4;
  c.nt = ceil(tiles, c.wc);
  const bool many = (long long)ceil(points, 32) * nPanels > 256;
  c.mt = windows == 1 && c.wc == 4 && many ? 2 : 1;
  c.rows = windows > 1 ? 16 : 16 * c.mt * (4 / c.wc);
  return c;
}

}  // namespace phx
