// F64 instantiation of the direct coupling transform (coupling_direct.hpp).
#include "coupling_direct.hpp"

namespace phx {
template void launch_coupling<double>(const CoupParams&, bool, hipStream_t);

// As few windows as fit: whole panels of up to 24 column tiles (FP32) or 12
// (FP64, whose tiles take twice the registers and LDS).  One column wave up to 3
// tiles, two up to 8, four beyond; the other waves take rows.  Several windows leave a row
// tile's g' in LDS between them, so they run 16 rows per workgroup.
CoupTiling coupling_tiling(bool f64, int nm, int nw, int nb2max) {
  CoupTiling c{};
  const size_t scratch = size_t(16) * nm * nb2max * (sizeof(double2) + sizeof(double));
  const int most = f64 ? 192 : 384;
  int windows = ceil_div(nm, std::max(1, most / nw));
  for (;; ++windows) {
    c.modes = ceil_div(nm, windows);
    windows = ceil_div(nm, c.modes);
    const size_t g3 = (size_t(16) * c.modes * nw * (f64 ? 16 : 8) + 15) / 16 * 16;
    c.stage = g3 >= size_t(16) * (nm + nb2max) * sizeof(double);
    c.lds = std::max(g3 + scratch, size_t(kGMax) * kCMax * 4 * sizeof(double));
    if (c.lds <= 160 * 1024 || c.modes == 1) break;
  }
  const int tiles = ceil_div(c.modes * nw, 16);
  c.wc = windows > 1 ? 4 : tiles <= 3 ? 1 : tiles <= 8 ? 2 : 4;
  c.nt = ceil_div(tiles, c.wc);
  c.mt = windows == 1 && c.wc == 4 ? 2 : 1;
  c.rows = windows > 1 ? 16 : 16 * c.mt * (4 / c.wc);
  return c;
}
}  // namespace phx
