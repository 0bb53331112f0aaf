// Which kernels run the last stage of the mesh-separable transform: one rule, for
// the buffers a batch reserves, the stages it launches and the column order they
// hand on.  Plain C++: no device code.
#pragma once

#include <cstddef>

namespace phx {

constexpr size_t kLdsBytes = 160 * 1024;  // of a workgroup
constexpr int kSplitCols = 4 * 6 * 16;    // widest panel of the split stage and of k_sep_xm: six tiles a wave
constexpr int kXgCols = 4 * 3 * 16;       // of k_sep_xg: three tiles a wave
constexpr int kSplitGroups = 24;          // x-groups whose 12 k-steps fit the x-stage's registers

// LDS of the y-stage (twiddles, quad entries, group ends) and of k_sep_yx.
constexpr size_t sep_y_lds_bytes(int my, int nQuads) {
  return size_t(my) * 16 + size_t(4) * nQuads * 8 + (size_t(nQuads) * sizeof(int) + 15) / 16 * 16;
}
constexpr size_t sep_yx_lds_bytes(int elem, int nQuads, int my, int nG0, int m0) {
  const int kp = (2 * nG0 + 3) / 4 * 4;
  return sep_y_lds_bytes(my, nQuads) + size_t(m0) * (kp + 1) * 2 * elem + size_t(16) * (kp * 16 + 16) * elem +
         size_t(4) * 64 * sizeof(int) + 64;
}

enum LastStage {
  kStageFused = 0,  // k_sep_y, then k_sep_xm (up to kSplitCols columns) or k_sep_x: x-stage and epilogue together
  kStageXg = 1,     // k_sep_y, k_sep_xg and k_sep_ep2: g3 rows through device memory
  kStageRot = 2,    // the same with the electron rotation in k_sep_xg: g' rows
  kStageYx = 3,     // k_sep_yx (the y-stage inside, no T2) and k_sep_ep2
};

struct LastStageSizes {
  int f64, bf16x3;    // data of the transform; split-BF16x3 x-stage
  int nm, nw;
  int m0, my;         // x and y mesh
  int nG0, nQuads;    // x-groups, y-stage quads
  int adaptive;       // adaptive smearing
};

// mode: phx_lw_set_split_last_stage's; fuseY: phx_lw_set_fused_y_stage's; learned: the
// learned screen's slot masks are used.
// Split: an x-stage kernel and an epilogue kernel write and read g3 but hide their
// latency at 2 to 4 waves per SIMD, where the fused kernel runs at 1 or 2: with 18
// modes x 16 bands in FP32 on a 32^3 mesh 7.2 against 21.8 ms per pass, 12 x 16 in
// FP64 on a 27 x 28 x 29 mesh 6.3 against 21.2.  It needs row masks of one word
// (m0 <= 64), an epilogue of 16 w2 (nw <= 16) and the x-stage's operands in registers
// (kSplitGroups, kSplitCols).  k_sep_yx takes both precisions but no slot masks;
// k_sep_xg FP32, 16 modes and kXgCols columns.
constexpr LastStage last_stage(const LastStageSizes& z, int mode, bool fuseY, bool learned) {
  if (!mode || z.bf16x3 || z.nw > 16 || z.m0 > 64 || z.nG0 > kSplitGroups || z.nm * z.nw > kSplitCols)
    return kStageFused;
  if (fuseY && !learned && mode != 3 && sep_yx_lds_bytes(z.f64 ? 8 : 4, z.nQuads, z.my, z.nG0, z.m0) <= kLdsBytes)
    return kStageYx;
  if (z.f64 || z.nm > 16 || z.nm * z.nw > kXgCols) return kStageFused;
  return mode == 3 && !z.adaptive ? kStageRot : kStageXg;
}

// Panels per launch of the split last stage when its g3 rows may take `room` bytes:
// between 16 and 128, as fewer, larger launches have shorter tails.
constexpr double kG3RoomMax = 24. * (1ull << 30);
constexpr double kG3Share = 0.25;  // of the memory that is free when the rows are made
constexpr int panel_chunk(double bytesPerPanel, double room) {
  const double n = room / bytesPerPanel;
  return n < 16. ? 16 : n > 128. ? 128 : int(n);
}

}  // namespace phx
