// Direct R_ph transform of the coupling with the shared epilogue (coupling_kernel.hpp),
// instantiated per precision in coupling_direct_f64.hip and coupling_direct_f32.hip.
#pragma once

#include "coupling_kernel.hpp"

namespace phx {

// g3(row, c) = sum_Rp A(Rp, row) C(Rp, c) as a complex product of real MFMAs: M
// = inner points, N = panel columns, K = R_p in quads, real and imaginary parts
// of g3 in accumulators of their own (Re += Ar x, Im += Ai x, Re += (-Ai) y, Im += Ar
// y for C = x + i y).  No LDS and no barrier in the main loop: a wave reads A (16
// lanes, consecutive points) and C (16 lanes, consecutive columns) straight into
// registers, two quads at a time, and every load of C serves four products per
// row tile.  The matrix cores bound it where nm nw fills the tiles; with C as a
// real [C; iC] panel and A staged in LDS between barriers one 4- or 8-byte load
// fed one product per row tile, and wide panels were bound by those loads.
// What is left is the epilogue's latency, and spills: the reduction's partial sums
// (64 registers) live through the main loop, so two row tiles spill 32, 71 and 102
// registers with 4, 5 and 6 column tiles in FP32 and 79 with 3 in FP64 (1 x 4: 8).
// Per launch: 48 columns, 251 R_p, 1700
// points, 32 outer points in FP64 0.23 -> 0.17 ms; 345 columns, 79 R_p in FP32
// 3.0 -> 2.2 ms.
template <typename T, int MT, int NT, bool REDUCE>
__global__ void __launch_bounds__(256, 2) k_coupling(CoupParams p, CoupTiling c) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef typename Vec2<T>::type T2;
  typedef typename Mfma4<T>::acc_t acc_t;
  constexpr int D = 2;
  const int nTilesTot = p.nPanels * p.nMtiles;
  const int bid = blockIdx.x;
  const int perXcd = gridDim.x / 8;
  const int L = (bid % 8) * perXcd + bid / 8;  // XCD-contiguous logical index
  if (L >= nTilesTot) return;
  const int panel = L / p.nMtiles, mtile = L % p.nMtiles;
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, lr = lane & 15,
            lg = lane >> 4;
  const int wc = wave % c.wc, wr = wave / c.wc;
  const int row0 = mtile * c.rows;
  const int kk = p.panelKK[panel];
  const int b1p = p.panelB1[panel];
  p.rowU2off += kk * p.rowKKStride;
  p.out += kk * p.outKKStride;
  const T2* A = static_cast<const T2*>(p.A);
  const T2* B = reinterpret_cast<const T2*>(static_cast<const T*>(p.B) + size_t(panel) * p.panelStride);
  const size_t ldb = size_t(p.ldb) / 2;
  int ar[MT];  // points beyond M read the last one; nothing uses their sums
#pragma unroll
  for (int m = 0; m < MT; ++m) ar[m] = min(row0 + (wr * MT + m) * 16 + lr, p.M - 1);
  T2* g3 = reinterpret_cast<T2*>(smem);  // 16 x window columns
  const int wcols = c.modes * p.nw;
  unsigned char* scratch = smem + (size_t(16) * wcols * sizeof(T2) + 15) / 16 * 16;
  const int nq = p.nRp / 4;
  double part[kGMax][kCMax];
#pragma unroll
  for (int gi = 0; gi < kGMax; ++gi)
#pragma unroll
    for (int k = 0; k < kCMax; ++k) part[gi][k] = 0.;

  for (int nu0 = 0; nu0 < p.nm; nu0 += c.modes) {
    const int nu1 = min(p.nm, nu0 + c.modes), cols = (nu1 - nu0) * p.nw;
    const T2* Bc[NT];  // columns beyond the window read its last one
#pragma unroll
    for (int j = 0; j < NT; ++j) Bc[j] = B + nu0 * p.nw + min((wc * NT + j) * 16 + lr, cols - 1);
    acc_t re[MT][NT], im[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) re[m][j][i] = im[m][j][i] = 0;
    T2 a[D][MT], b[D][NT];
    auto load = [&](T2(&aa)[MT], T2(&bb)[NT], int q) {
      const int r = 4 * q + lg;
      const size_t rb = size_t(min(r, p.nRp - 1)) * ldb;
#pragma unroll
      for (int j = 0; j < NT; ++j) bb[j] = Bc[j][rb];
#pragma unroll
      for (int m = 0; m < MT; ++m) aa[m] = A[size_t(r) * p.lda + ar[m]];
    };
    auto product = [&](const T2(&aa)[MT], const T2(&bb)[NT]) {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          re[m][j] = Mfma4<T>::mac(aa[m].x, bb[j].x, re[m][j]);
          im[m][j] = Mfma4<T>::mac(aa[m].y, bb[j].x, im[m][j]);
        }
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          re[m][j] = Mfma4<T>::mac(-aa[m].y, bb[j].y, re[m][j]);
          im[m][j] = Mfma4<T>::mac(aa[m].x, bb[j].y, im[m][j]);
        }
    };
    const int qLast = max(nq - 1, 0);
#pragma unroll
    for (int d = 0; d < D; ++d) load(a[d], b[d], min(d, qLast));
    int i = 0;
    for (; i + D <= nq; i += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        product(a[d], b[d]);
        load(a[d], b[d], min(i + d + D, qLast));  // unconditional: see k_cache
      }
    }
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
      if (i + d < nq) product(a[d], b[d]);
    if (p.nRp & 3) {  // the last R_p, less than a quad
      load(a[0], b[0], nq);
      if (4 * nq + lg >= p.nRp)
#pragma unroll
        for (int j = 0; j < NT; ++j) b[0][j] = T2{T(0), T(0)};
      product(a[0], b[0]);
    }
    // 16 rows at a time into LDS, then the epilogue by all threads
    const int tiles = c.rows / 16;
    for (int h = 0; h < tiles; ++h) {
      if (row0 + 16 * h >= p.M) break;
      __syncthreads();
#pragma unroll
      for (int m = 0; m < MT; ++m)
        if (wr * MT + m == h)
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            const int col = (wc * NT + j) * 16 + lr;
            if (col < cols)
#pragma unroll
              for (int k = 0; k < 4; ++k) g3[Mfma4<T>::row(lg, k) * wcols + col] = T2{re[m][j][k], im[m][j][k]};
          }
      __syncthreads();
      const int row = row0 + 16 * h + (t >> 4);
      const int myRow = row < p.M ? row : -1;
      epilogue16_u2<T>(p, reinterpret_cast<const T*>(g3), 2 * wcols, scratch, myRow, nu0, nu1);
      if (nu1 < p.nm) continue;  // several windows: one row tile (rows = 16)
      __syncthreads();
      int myIq = 0;
      if (myRow >= 0)
        myIq = p.qmode ? mesh_diff_index(p.rowMesh[myRow], p.kkMesh[kk], p.m0, p.m1, p.m2) : p.rowE3[myRow];
      epilogue16_tail<REDUCE>(p, scratch, c.stage ? reinterpret_cast<double*>(g3) : nullptr, panel, kk, b1p, myRow, myIq, part);
    }
  }
  if (REDUCE) reduce_partials<kCMax>(p, L, smem, part);
}

template <typename T>
void launch_coupling(const CoupParams& p, bool reduce, hipStream_t s) {
  PHX_REQUIRE(p.nm <= kNmMax, "coupling kernel supports nm <= 36");
  PHX_REQUIRE(p.ldb % 2 == 0 && p.nRp >= 1 && p.lda >= size_t(std::max(p.M, 1)), "coupling kernel: bad operand shapes");
  const CoupTiling c = coupling_tiling(sizeof(T) == 8, p.nm, p.nw, p.nb2max, p.M, p.nPanels);
  PHX_REQUIRE(c.lds <= 160 * 1024, "coupling kernel: nm x bands per inner point too large for LDS");
  PHX_REQUIRE(p.nMtiles == ceil_div(p.M, c.rows), "coupling kernel: row tiles");
  const int tiles = p.nPanels * p.nMtiles;
  if (tiles <= 0) return;
  auto go = [&](auto kern) {
    PHX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                int(c.lds)));
    hipLaunchKernelGGL(kern, dim3(ceil_div(tiles, 8) * 8), dim3(256), c.lds, s, p, c);
  };
  // the tiles per wave that coupling_tiling gives: FP64 at most 4 columns (3 with two row tiles)
  auto red = [&](auto mt, auto nt) {
    constexpr int MT = decltype(mt)::value, NT = decltype(nt)::value;
    if constexpr (MT == 1 ? NT <= (sizeof(T) == 8 ? 4 : 6) : NT >= 3 && NT <= (sizeof(T) == 8 ? 3 : 6)) {
      if (reduce) go(k_coupling<T, MT, NT, true>);
      else go(k_coupling<T, MT, NT, false>);
    } else {
      PHX_REQUIRE(false, "coupling kernel: no instance for these tiles");
    }
  };
  auto nts = [&](auto mt) {
    switch (c.nt) {
      case 1: red(mt, std::integral_constant<int, 1>{}); break;
      case 2: red(mt, std::integral_constant<int, 2>{}); break;
      case 3: red(mt, std::integral_constant<int, 3>{}); break;
      case 4: red(mt, std::integral_constant<int, 4>{}); break;
      case 5: red(mt, std::integral_constant<int, 5>{}); break;
      default: red(mt, std::integral_constant<int, 6>{});
    }
  };
  if (c.mt == 1) nts(std::integral_constant<int, 1>{});
  else nts(std::integral_constant<int, 2>{});
  PHX_HIP(hipGetLastError());
}

}  // namespace phx
