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
// where g' and |g|^2 of a row tile leave less LDS to g3: half of the LDS, for two
// workgroups per CU, where there are more than 256 and a window keeps a quarter of
// its modes (27 modes x 19 bands in FP32, 4 bands per point, 1888 workgroups of 32
// points: 1490 us with one workgroup per CU, 946 with two).  Several windows leave a
// row tile's g' in LDS between them, so they run 16 rows per workgroup.
// Whole panels take 16, 32 or 64 rows: more rows share a load of the panel, but
// their epilogues follow each other, and two workgroups per CU, 512 in all, run at
// once.  16 rows on four column waves while 32 would not even give every CU a
// workgroup.  Else, up to 8 column tiles, 64 rows where they take less time than
// 32: a workgroup of 64 takes 1.6 times as long as one of 32 (6 to 8 tiles 1.75), a
// launch as long as its workgroups of 512 at once, at least one such wave, two beyond
// 512 of 32 rows, and 0.3 waves for the tail of 64.  They run on one column wave up to
// 6 tiles (FP64, whose accumulators take twice the registers: 4), in FP32 on two with
// two row tiles each beyond.  More tiles: two row tiles on four column waves.
// us per launch with 16, 32 and 64 rows in FP32; 5 column tiles: 28 workgroups of 32
// rows 35, 52 and 63, 756 -, 108 and 97, 1022 -, 135 and 141, 12298 -, 1468 and 1230; 3
// tiles, 28: 27, 41 and 63; 8 tiles, 15738: -, 2389 and 2112.  18 tiles with 16
// and 32 rows: 108 workgroups of 32 rows 55 and 81, 256 64 and 83, 432 120 and 114,
// 3348 730 and 644.
inline CoupTiling coupling_tiling(bool f64, int nm, int nw, int nb2max, int points, int nPanels) {
  auto ceil = [](int a, int b) { return (a + b - 1) / b; };
  CoupTiling c{};
  const size_t scratch = size_t(16) * nm * nb2max * (16 + 8);
  const int most = f64 ? 192 : 384;
  const int whole = ceil(nm, ceil(nm, std::max(1, most / nw)));
  auto wgs = [&](int rows) { return (long long)ceil(points, rows) * nPanels; };
  auto tile = [&](int modes) { return (size_t(16) * modes * nw * (f64 ? 16 : 8) + 15) / 16 * 16; };
  auto lds = [&](int modes) { return std::max(tile(modes) + scratch, kCoupReduceLds); };
  auto fit = [&](size_t room) {
    int modes = whole;
    // even windows, and at least one mode less: ceil(nm / (windows + 1)) can be the same number of modes
    while (modes > 1 && lds(modes) > room) modes = std::min(modes - 1, ceil(nm, ceil(nm, modes) + 1));
    return modes;
  };
  c.modes = fit(80 * 1024);
  if (wgs(16) <= 256 || lds(c.modes) > 80 * 1024 || 4 * c.modes < whole) c.modes = fit(160 * 1024);
  const int windows = ceil(nm, c.modes);
  c.stage = tile(c.modes) >= size_t(16) * (nm + nb2max) * 8;
  c.lds = lds(c.modes);
  const int tiles = ceil(c.modes * nw, 16);
  c.mt = 1;
  if (windows > 1 || wgs(32) <= 256) {
    c.wc = 4;
  } else if (tiles > 8) {
    c.wc = 4;
    c.mt = 2;
  } else {
    const long long t64 = wgs(64) <= 512 ? 512 : wgs(64) + 154;
    const long long t32 = wgs(32) <= 512 ? 512 : std::max(wgs(32), 1024ll);
    const bool tall = tiles <= 5 ? 8 * t64 <= 5 * t32 : 7 * t64 <= 4 * t32;
    c.wc = tall && tiles <= (f64 ? 4 : 6) ? 1 : 2;
    c.mt = tall && !f64 && tiles > 6 ? 2 : 1;
  }
  c.nt = ceil(tiles, c.wc);
  c.rows = windows > 1 ? 16 : 16 * c.mt * (4 / c.wc);
  return c;
}

}  // namespace phx
