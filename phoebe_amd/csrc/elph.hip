// Electron-phonon coupling kernels: InteractionElPhWan::cacheElPh and
// calcCouplingSquared (interaction_elph.cpp:229-448, 492-701) plus the
// Gaussian-delta linewidth reduction of ElScatteringMatrix::builder
// (el_scattering.cpp:216-386), re-designed for gfx950.
//
// Data flow for one batch of outer points k1 (index kk inside the batch):
//
//  k_cache   g1(Rp,nu,w1,w2) = sum_Re e^{ik1.Re}/de gW(Re,Rp,nu,w1,w2)   [k1-batched: every
//            gW element is read once per batch and used for every k1]
//            C(Rp,nu,b1,w2) = sum_w1 g1 U1(w1,b1) * s(k1,Rp)               [fused epilogue]
//            with s = e^{-ik1.Rp}/dp (mesh mode) or 1/dp (explicit-q mode), written
//            as complex panels (Rp, (nu, w2)), one panel per (k1, b1).
//  k_coupling  rows = outer-product partners (k2 or explicit q):
//            g3(row, nu, w2) = sum_Rp A(row, Rp) C(Rp, nu, b1, w2)            [MFMA,
//            A(row, .) = e^{ik2.Rp}, so e^{iq.Rp} = e^{ik2.Rp} e^{-ik1.Rp}]
//            epilogue in LDS: g4 = e3^T g3 (phonon rotation, e3 not conjugated),
//            g = U2^H g4, |g|^2, then either store |g|^2 (calcCouplingSquared) or
//            symmetrize over degenerate b2 / nu groups and contract with the
//            Gaussian-delta weights into per-workgroup partial linewidths.
//  k_collect  sums the partials in a fixed order (deterministic, no float atomics),
//            including the b1 degenerate-group average of symmetrizeCoupling.
#include <algorithm>
#include <thread>
#include <type_traits>
#include <vector>

#include "elph_params.hpp"
#include "phx_common.hpp"

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));

namespace phx {

// ------------------------------------------------------------------ synthetic gW
__host__ __device__ inline uint64_t mix64(uint64_t x) {
  x ^= x >> 30;
  x *= 0xBF58476D1CE4E5B9ull;
  x ^= x >> 27;
  x *= 0x94D049BB133111EBull;
  x ^= x >> 31;
  return x;
}
__host__ __device__ inline double hash_u(uint64_t seed, uint64_t ctr) {
  uint64_t h = mix64(seed + ctr * 0x9E3779B97F4A7C15ull);
  return double(h >> 11) * (1.0 / 9007199254740992.0);
}
__host__ __device__ inline double hash_n(uint64_t seed, uint64_t idx) {
  uint64_t c = idx * 4;
  double s = hash_u(seed, c) + hash_u(seed, c + 1);
  s = s + hash_u(seed, c + 2);
  s = s + hash_u(seed, c + 3);
  return (s - 2.0) * 1.7320508075688772;
}

template <typename T2>
__global__ void k_synth_gw(T2* __restrict__ gW, size_t n, size_t blk,
                           const double* __restrict__ decay, uint64_t seed) {
  for (size_t f = size_t(blockIdx.x) * blockDim.x + threadIdx.x; f < n;
       f += size_t(gridDim.x) * blockDim.x) {
    double d = decay[f / blk];
    T2 v;
    v.x = d * hash_n(seed, 2 * f);
    v.y = d * hash_n(seed, 2 * f + 1);
    gW[f] = v;
  }
}

void synth_gw_host(double* gW, size_t n, size_t blk, const double* decay, uint64_t seed) {
  unsigned nt = std::max(1u, std::min(32u, std::thread::hardware_concurrency()));
  std::vector<std::thread> th;
  for (unsigned t = 0; t < nt; ++t)
    th.emplace_back([=] {
      for (size_t f = t; f < n; f += nt) {
        double d = decay[f / blk];
        gW[2 * f] = d * hash_n(seed, 2 * f);
        gW[2 * f + 1] = d * hash_n(seed, 2 * f + 1);
      }
    });
  for (auto& x : th) x.join();
}

void launch_synth_gw(double2* gW, size_t n, size_t blk, const double* decay, uint64_t seed,
                     hipStream_t s) {
  hipLaunchKernelGGL(k_synth_gw<double2>, dim3(8192), dim3(256), 0, s, gW, n, blk, decay, seed);
  PHX_HIP(hipGetLastError());
}

// FP32 copy of the same tensor, each element rounded once from its FP64 value.
void launch_synth_gw_f32(float2* gW, size_t n, size_t blk, const double* decay, uint64_t seed,
                         hipStream_t s) {
  hipLaunchKernelGGL(k_synth_gw<float2>, dim3(8192), dim3(256), 0, s, gW, n, blk, decay, seed);
  PHX_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ small kernels
template <typename T>
__global__ void k_fill(T* p, size_t n, T v) {
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += size_t(gridDim.x) * blockDim.x)
    p[i] = v;
}

template <typename T>
void launch_fill(T* p, size_t n, T v, hipStream_t s) {
  if (!n) return;
  int blocks = int(std::min<size_t>(8192, (n + 255) / 256));
  hipLaunchKernelGGL(k_fill<T>, dim3(blocks), dim3(256), 0, s, p, n, v);
  PHX_HIP(hipGetLastError());
}
template void launch_fill<double>(double*, size_t, double, hipStream_t);
template void launch_fill<float>(float*, size_t, float, hipStream_t);
template void launch_fill<int>(int*, size_t, int, hipStream_t);

// Phase table P(i, r) = e^{sign i k_i.R_r} * scale_r  (double2, rows x nR).
__global__ void k_phase_table(int rows, int nR, const double* __restrict__ kc,
                              const double* __restrict__ R, const double* __restrict__ scale,
                              double sign, double2* __restrict__ P) {
  size_t n = size_t(rows) * nR;
  for (size_t t = size_t(blockIdx.x) * blockDim.x + threadIdx.x; t < n;
       t += size_t(gridDim.x) * blockDim.x) {
    int i = int(t / nR), r = int(t % nR);
    double arg = kc[3 * i] * R[3 * r] + kc[3 * i + 1] * R[3 * r + 1] + kc[3 * i + 2] * R[3 * r + 2];
    double s, c;
    sincos(arg, &s, &c);
    double sc = scale ? scale[r] : 1.0;
    P[t] = make_double2(c * sc, sign * s * sc);
  }
}

void launch_phase_table(int rows, int nR, const double* kc, const double* R, const double* scale,
                        double sign, double2* P, hipStream_t s) {
  if (rows <= 0) return;
  hipLaunchKernelGGL(k_phase_table, dim3(4096), dim3(256), 0, s, rows, nR, kc, R, scale, sign, P);
  PHX_HIP(hipGetLastError());
}

// The same table transposed for the GEMMs of k_cache and k_coupling, in their
// precision: out(r, i) with `cols` >= rows points per row (points beyond `rows`
// zero) and nR rounded up to whole quads (rows beyond nR zero).
template <typename T>
__global__ void k_phase_cols(int rows, int cols, int nR, const double* __restrict__ kc,
                             const double* __restrict__ R, const double* __restrict__ scale, T* __restrict__ out) {
  const size_t n = size_t(nR + 3) / 4 * 4 * cols;
  for (size_t t = size_t(blockIdx.x) * blockDim.x + threadIdx.x; t < n; t += size_t(gridDim.x) * blockDim.x) {
    const int r = int(t / cols), i = int(t - size_t(r) * cols);
    double s = 0., c = 0.;
    if (r < nR && i < rows) {
      sincos(kc[3 * i] * R[3 * r] + kc[3 * i + 1] * R[3 * r + 1] + kc[3 * i + 2] * R[3 * r + 2], &s, &c);
      if (scale) {
        s *= scale[r];
        c *= scale[r];
      }
    }
    out[2 * t] = T(c);
    out[2 * t + 1] = T(s);
  }
}

template <typename T>
void launch_phase_cols(int rows, int cols, int nR, const double* kc, const double* R, const double* scale, void* out,
                       hipStream_t s) {
  if (rows <= 0) return;
  const size_t n = phase_cols_size(nR, cols);
  hipLaunchKernelGGL(k_phase_cols<T>, dim3(unsigned(std::min<size_t>((n + 255) / 256, 16384))), dim3(256), 0, s, rows,
                     cols, nR, kc, R, scale, static_cast<T*>(out));
  PHX_HIP(hipGetLastError());
}
template void launch_phase_cols<double>(int, int, int, const double*, const double*, const double*, void*, hipStream_t);
template void launch_phase_cols<float>(int, int, int, const double*, const double*, const double*, void*, hipStream_t);

// Gather windowed eigenvector columns: pool(off_a + w + nw*b) = U(ik_a)(w, lo_a + b).
__global__ void k_gather_eig(int na, int nw, const int* __restrict__ ik, const int* __restrict__ lo,
                             const int* __restrict__ nb, const int* __restrict__ off,
                             const double2* __restrict__ U, double2* __restrict__ pool) {
  int a = blockIdx.x;
  if (a >= na) return;
  int n = nb[a] * nw;
  const double2* src = U + size_t(ik[a]) * nw * nw + size_t(lo[a]) * nw;
  for (int t = threadIdx.x; t < n; t += blockDim.x) pool[off[a] + t] = src[t];
}

void launch_gather_eig(int na, int nw, const int* ik, const int* lo, const int* nb, const int* off,
                       const double2* U, double2* pool, hipStream_t s) {
  if (na <= 0) return;
  hipLaunchKernelGGL(k_gather_eig, dim3(na), dim3(256), 0, s, na, nw, ik, lo, nb, off, U, pool);
  PHX_HIP(hipGetLastError());
}

// Scatter phonon results of a compact q list into full-mesh indexed tables.
__global__ void k_scatter_ph(int nq, int nm, const int* __restrict__ iq, const double* __restrict__ w,
                             const double2* __restrict__ ev, double* __restrict__ wAll,
                             double2* __restrict__ evAll) {
  int j = blockIdx.x;
  if (j >= nq) return;
  int q = iq[j];
  for (int t = threadIdx.x; t < nm * nm; t += blockDim.x)
    evAll[size_t(q) * nm * nm + t] = ev[size_t(j) * nm * nm + t];
  for (int t = threadIdx.x; t < nm; t += blockDim.x) wAll[size_t(q) * nm + t] = w[size_t(j) * nm + t];
}

void launch_scatter_ph(int nq, int nm, const int* iq, const double* w, const double2* ev,
                       double* wAll, double2* evAll, hipStream_t s) {
  if (nq <= 0) return;
  hipLaunchKernelGGL(k_scatter_ph, dim3(nq), dim3(256), 0, s, nq, nm, iq, w, ev, wAll, evAll);
  PHX_HIP(hipGetLastError());
}

// Phonon eigenvectors of every q in the layout the separable transform's
// epilogue reads, in its precision: out(q)(nu, nu2) at nu * nm + nu2, i.e.
// the lanes that serve the modes nu2 of one row read consecutive elements.
template <typename T2v>
__global__ void k_transpose_e3(int nk, int nm, const double2* __restrict__ ev, T2v* __restrict__ out) {
  const int q = blockIdx.x;
  if (q >= nk) return;
  const size_t base = size_t(q) * nm * nm;
  for (int t = threadIdx.x; t < nm * nm; t += blockDim.x) {
    const int nu = t / nm, nu2 = t % nm;
    const double2 e = ev[base + nu + size_t(nm) * nu2];
    out[base + t] = T2v{decltype(out->x)(e.x), decltype(out->x)(e.y)};
  }
}

void launch_transpose_e3(int nk, int nm, const double2* ev, void* out, bool fp32, hipStream_t s) {
  if (nk <= 0) return;
  if (fp32)
    hipLaunchKernelGGL(k_transpose_e3<float2>, dim3(nk), dim3(256), 0, s, nk, nm, ev,
                       static_cast<float2*>(out));
  else
    hipLaunchKernelGGL(k_transpose_e3<double2>, dim3(nk), dim3(256), 0, s, nk, nm, ev,
                       static_cast<double2*>(out));
  PHX_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ cacheElPh
// g1(k1; Rp,nu,w1,w2) = sum_Re P(k1,Re) gW(Re,Rp,nu,w1,w2) as a real MFMA GEMM:
// M = the outer points (tiles of 16, real and imaginary parts of g1 in
// accumulators of their own), N = gW columns, K = R_e in quads.  Lane (lr, lg)
// loads P(R_e = 4q + lg, point lr) and gW(R_e, column lr) as complex numbers,
// and four products per tile pair and quad take their components:
//   Re += Pr x, Im += Pi x;  Re += (-Pi) y, Im += Pr y     (gW = x + i y).
// A workgroup owns whole (Rp, nu) blocks of nw^2 columns, so the U1 rotation
// and the e^{-ik1.Rp}/dp factor run as its epilogue.

template <typename T> struct Vec2;
template <> struct Vec2<double> { typedef double2 type; };
template <> struct Vec2<float> { typedef float2 type; };

template <typename T> struct MfmaC;
template <> struct MfmaC<double> {
  typedef d4_t acc_t;
  __device__ static acc_t mac(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static int row(int lk, int i) { return lk + 4 * i; }
};
template <> struct MfmaC<float> {
  typedef f4_t acc_t;
  __device__ static acc_t mac(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static int row(int lk, int i) { return 4 * lk + i; }
};

// Panel epilogue of k_cache.  Cb holds g1 of up to 16 outer points (in rows
// 0..15 the real parts, in rows 16..31 the imaginary parts, CW elements per row)
// for the columns (w1, w2), w1lo <= w1 < w1hi, of the nblk blocks (rp, nu) from blk0
// on, one after the other; pan[0 .. np - 1] are those points' panels: (row in Cb | point << 4, offset of its U1 column).
// Applies the U1 rotation over that w1 range and the factor s(k1, Rp), and
// writes (w1lo == 0) or adds (later passes) the panel entries.  Each output
// (panel, w2) is owned by the same thread in every pass (the thread-to-output
// map does not depend on w1lo).
// All blocks of the workgroup in one loop: at nw = 1 it holds 64 of them, and one
// after the other with a thread per panel they took 72 us of a batch of 32 points
// (FP32, 3 modes, 10 x 11 x 9 mesh), 19 so.
template <typename T, typename OutT>
__device__ __forceinline__ void cache_panel_epilogue(const CacheParams& p, const T* Cb, int CW, int w1lo, int w1hi,
                                                     const int2* pan, int pan0, int np, int blk0, int nblk) {
  typedef typename Vec2<OutT>::type O2;
  const int nw = p.nw, per = np * nw;
  for (int idx = threadIdx.x; idx < nblk * per; idx += 256) {
    const int bl = nblk > 1 ? idx / per : 0, rest = idx - bl * per;
    const int e = rest / nw, w2 = rest - e * nw, rp = (blk0 + bl) / p.nm, nu = (blk0 + bl) - rp * p.nm;
    const int2 m = pan[e];
    const int kl = m.x & 15;
    const double2 s = p.phP[size_t(m.x >> 4) * p.nRp + rp];
    const double2* U1 = p.U1pool + m.y;
    const T* xr = Cb + kl * CW + bl * nw * nw + w2 - w1lo * nw;
    const T* xi = xr + 16 * CW;
    double2 v = make_double2(0., 0.);
#pragma unroll 8
    for (int w1 = w1lo; w1 < w1hi; ++w1) {
      const double ar = double(xr[w1 * nw]), ai = double(xi[w1 * nw]);
      const double2 u = U1[w1];
      v.x += ar * u.x - ai * u.y;
      v.y += ar * u.y + ai * u.x;
    }
    const double2 c = make_double2(v.x * s.x - v.y * s.y, v.x * s.y + v.y * s.x);
    O2* out = reinterpret_cast<O2*>(static_cast<OutT*>(p.B) + size_t(pan0 + e) * p.panelStride + size_t(rp) * p.ldb) +
              size_t(nu) * nw + w2;
    if (w1lo == 0) out[0] = O2{OutT(c.x), OutT(c.y)};
    else out[0] = O2{out[0].x + OutT(c.x), out[0].y + OutT(c.y)};  // later column passes add their w1 range
  }
}

// How k_cache cuts the gW columns: a workgroup takes `blocks` whole (Rp, nu)
// blocks of nw^2 columns in `passes` passes of `w1Rows` rows of nw columns, as
// ntw tiles of 16 columns per wave on wc waves; 4 / wc waves share the R_e sum.
struct CacheTiling {
  int blocks, passes, w1Rows, wc, ntw;
};
inline CacheTiling cache_tiling(int nw) {
  CacheTiling t{};
  const int E = nw * nw;
  t.blocks = E <= 32 ? 64 / E : 1;
  t.passes = t.blocks > 1 ? 1 : (nw + 256 / nw - 1) / (256 / nw);
  t.w1Rows = (nw + t.passes - 1) / t.passes;
  const int cols = t.blocks > 1 ? t.blocks * E : t.w1Rows * nw;
  const int tiles = (cols + 15) / 16;
  t.wc = tiles <= 4 ? 1 : tiles <= 8 ? 2 : 4;
  t.ntw = (tiles + t.wc - 1) / t.wc;
  return t;
}
// LDS row of the epilogue (elements): every column of the pass, padded so that
// the four row groups of an accumulator tile fall into different banks.
__host__ __device__ inline int cache_row(int wc, int ntw) { return 16 * wc * ntw + 4; }

// Bound by HBM and the matrix cores alike at a batch of 32 points (16 bytes and
// 256 FLOP per gW element in FP64), by HBM at a few points.  The main loop has
// no barrier: a wave reads its A fragment (the phases, transposed so that 16
// lanes read consecutive points; a table of some 100 KB that stays in L2) and
// its gW columns straight into registers, two R_e quads at a time.  With few
// columns per block (nw <= 11) two or all four waves of a workgroup share the
// block and split the R_e sum, which LDS adds up in wave order; with all four on
// columns, three of them had none at nw = 8.  A batch of up to 16 points runs
// one tile of points instead of two.
// nw = 8, 6 modes, R on WS(7^3) x WS(6^3) (0.73 GB of gW in FP64), against a
// version with the phases staged in LDS between barriers and all waves on
// columns: 32 points 0.98 -> 0.22 ms in FP64 (52 TFLOP/s) and 0.55 -> 0.145 ms
// in FP32; one point 0.89 -> 0.16 ms (4.6 TB/s, the copy rate).
template <typename T, typename OutT, int MH, int NTW>
__global__ void __launch_bounds__(256, MH * sizeof(T) > 16 ? 1 : 2) k_cache(CacheParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef typename Vec2<T>::type T2;
  typedef typename MfmaC<T>::acc_t acc_t;
  constexpr int D = 2;  // 3 and 4 cost FP32 registers and time
  const int E = p.nw * p.nw, nBlocks = p.nRp * p.nm;
  const int blk0 = blockIdx.x * p.blocks, nblk = min(p.blocks, nBlocks - blk0);
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, lr = lane & 15, lg = lane >> 4;
  const int WC = p.wc, WK = 4 / WC, wc = wave % WC, wk = wave / WC;
  const int CW = cache_row(WC, NTW);
  T* Cb = reinterpret_cast<T*>(smem);  // (WK, 32, CW): real parts of 16 points, then imaginary
  int2* sPan = reinterpret_cast<int2*>(Cb + size_t(WK) * 32 * CW);  // the job's panels
  const size_t stride = size_t(nBlocks) * E;
  // the job: rows summed over (R_e of gW, or the groups of a line's Tg), their
  // phase table and the outer points kk0 .. kk0 + nk - 1
  const int4 jb = p.jobs ? p.jobs[blockIdx.y] : make_int4(0, p.nkk, 0, 0);
  const int kk0 = jb.x, nk = jb.y, nRows = p.jobs ? p.nGe : p.nRe;
  const T2* G = (p.jobs ? static_cast<const T2*>(p.Tg) + size_t(jb.z) * nRows * stride : static_cast<const T2*>(p.gW)) +
                size_t(blk0) * E;
  const T2* ph = static_cast<const T2*>(p.phE) + size_t(blockIdx.y) * ((nRows + 3) / 4 * 4) * (16 * MH);
  // the panels' metadata goes to LDS while the main loop runs: read in the
  // epilogue, its chain of loads took longer there than the products
  const int pan0 = p.panelBase[kk0];
  for (int i = t; i < nk * p.nb1Max; i += 256) {
    const int kl = i / p.nb1Max, b1 = i - kl * p.nb1Max, kk = kk0 + kl;
    if (b1 < p.nb1[kk]) sPan[p.panelBase[kk] - pan0 + b1] = make_int2(kk << 4 | (kl & 15), p.U1off[kk] + p.nw * b1);
  }
  const int nq = nRows / 4, q0 = nq * wk / WK, q1 = nq * (wk + 1) / WK;

  for (int w1lo = 0; w1lo < p.nw; w1lo += p.w1Rows) {
    const int w1hi = min(p.nw, w1lo + p.w1Rows);
    const int cols = p.blocks > 1 ? nblk * E : (w1hi - w1lo) * p.nw;
    const T2* Gc[NTW];  // columns beyond the pass read its last one; nothing uses their sums
#pragma unroll
    for (int j = 0; j < NTW; ++j) Gc[j] = G + size_t(w1lo) * p.nw + min((wc * NTW + j) * 16 + lr, cols - 1);
    acc_t accr[MH][NTW], acci[MH][NTW];
#pragma unroll
    for (int m = 0; m < MH; ++m)
#pragma unroll
      for (int j = 0; j < NTW; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) accr[m][j][i] = acci[m][j][i] = 0;
    // A ring of D quads.  The loop's loads are unconditional (quads beyond the
    // wave's last read valid rows again and are not used): a load under a branch
    // makes the compiler wait for every load in flight.
    T2 b[D][NTW], a[D][MH];
    auto load = [&](T2(&bb)[NTW], T2(&aa)[MH], int q) {
      const int re = 4 * q + lg;
      const size_t row = size_t(min(re, nRows - 1)) * stride;
#pragma unroll
      for (int j = 0; j < NTW; ++j) bb[j] = Gc[j][row];
#pragma unroll
      for (int m = 0; m < MH; ++m) aa[m] = ph[size_t(re) * (16 * MH) + 16 * m + lr];
    };
    auto product = [&](const T2(&bb)[NTW], const T2(&aa)[MH]) {
#pragma unroll
      for (int j = 0; j < NTW; ++j)
#pragma unroll
        for (int m = 0; m < MH; ++m) {
          accr[m][j] = MfmaC<T>::mac(aa[m].x, bb[j].x, accr[m][j]);
          acci[m][j] = MfmaC<T>::mac(aa[m].y, bb[j].x, acci[m][j]);
        }
#pragma unroll
      for (int j = 0; j < NTW; ++j)
#pragma unroll
        for (int m = 0; m < MH; ++m) {
          accr[m][j] = MfmaC<T>::mac(-aa[m].y, bb[j].y, accr[m][j]);
          acci[m][j] = MfmaC<T>::mac(aa[m].x, bb[j].y, acci[m][j]);
        }
    };
    const int n = q1 - q0, qLast = max(nq - 1, 0);
#pragma unroll
    for (int d = 0; d < D; ++d) load(b[d], a[d], min(q0 + d, qLast));
    int i = 0;
    for (; i + D <= n; i += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        product(b[d], a[d]);
        load(b[d], a[d], min(q0 + i + d + D, qLast));
      }
    }
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
      if (i + d < n) product(b[d], a[d]);
    if ((nRows & 3) && wk == WK - 1) {  // the last R_e, less than a quad: rows beyond them are zero
      load(b[0], a[0], nq);
      if (4 * nq + lg >= nRows)
#pragma unroll
        for (int j = 0; j < NTW; ++j) b[0][j] = T2{T(0), T(0)};
      product(b[0], a[0]);
    }
    // panel epilogue in passes of 16 outer points
#pragma unroll
    for (int m = 0; m < MH; ++m) {
      if (16 * m >= nk) break;
      __syncthreads();  // the previous pass has read Cb
      T* Cw = Cb + size_t(wk) * 32 * CW;
#pragma unroll
      for (int j = 0; j < NTW; ++j) {
        const int cl = (wc * NTW + j) * 16 + lr;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = MfmaC<T>::row(lg, i);
          Cw[r * CW + cl] = accr[m][j][i];
          Cw[(16 + r) * CW + cl] = acci[m][j][i];
        }
      }
      __syncthreads();
      if (WK > 1) {
        for (int i = t; i < 32 * CW; i += 256) {
          T v = Cb[i];
          for (int k = 1; k < WK; ++k) v += Cb[size_t(k) * 32 * CW + i];
          Cb[i] = v;
        }
        __syncthreads();
      }
      const int kl1 = min(16 * m + 16, nk) - 1;
      const int e0 = p.panelBase[kk0 + 16 * m] - pan0, e1 = p.panelBase[kk0 + kl1] + p.nb1[kk0 + kl1] - pan0;
      cache_panel_epilogue<T, OutT>(p, Cb, CW, w1lo, w1hi, sPan + e0, pan0 + e0, e1 - e0, blk0, nblk);
    }
  }
}

// tiles: 16-point tiles of the phase table's rows; nJobs: grid rows.
template <typename T, typename OutT>
static void launch_cache_gemm(CacheParams p, int tiles, int nJobs, hipStream_t s) {
  const CacheTiling c = cache_tiling(p.nw);
  p.blocks = c.blocks;
  p.w1Rows = c.w1Rows;
  p.wc = c.wc;
  PHX_REQUIRE(p.nb1Max >= 1 && p.nb1Max <= p.nw && p.ldb % 2 == 0, "cacheElPh kernel: bad band count or panel row");
  const size_t lds = size_t(4 / c.wc) * 32 * cache_row(c.wc, c.ntw) * sizeof(T) +
                     size_t(16) * tiles * p.nb1Max * sizeof(int2);
  auto go = [&](auto kern) {
    PHX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
    hipLaunchKernelGGL(kern, dim3(ceil_div(p.nRp * p.nm, c.blocks), nJobs), dim3(256), lds, s, p);
  };
  auto ntw = [&](auto mh) {
    constexpr int MH = decltype(mh)::value;
    switch (c.ntw) {
      case 1: go(k_cache<T, OutT, MH, 1>); break;
      case 2: go(k_cache<T, OutT, MH, 2>); break;
      case 3: go(k_cache<T, OutT, MH, 3>); break;
      default: go(k_cache<T, OutT, MH, 4>);
    }
  };
  if (tiles == 1) ntw(std::integral_constant<int, 1>{});
  else if (tiles == 2) ntw(std::integral_constant<int, 2>{});
  else ntw(std::integral_constant<int, 3>{});
  PHX_HIP(hipGetLastError());
}

template <typename T, typename OutT>
void launch_cache(const CacheParams& p, hipStream_t s) {
  PHX_REQUIRE(p.nw <= 32, "cacheElPh kernel supports nw <= 32");
  PHX_REQUIRE(p.nkk <= kCacheNKK, "cacheElPh kernel: too many outer points per launch");
  PHX_REQUIRE(!p.jobs, "cacheElPh kernel: jobs belong to the line form");
  if (p.nkk <= 0) return;
  launch_cache_gemm<T, OutT>(p, cache_phase_cols(p.nkk) / 16, 1, s);
}
template void launch_cache<double, double>(const CacheParams&, hipStream_t);
template void launch_cache<float, float>(const CacheParams&, hipStream_t);

// ------------------------------------------------------------------ cacheElPh on mesh lines
// Outer points that share the mesh line (j1, j2) and differ in j0 factor the
// phase: with n_d = b_d.R_e / 2pi,
//   e^{ik1.R_e} = e^{2 pi i j0 n0/m0} e^{2 pi i (j1 n1/m1 + j2 n2/m2)}.
// Stage a (one HBM stream over gW for up to kLinesPerBatch = 16 lines):
//   Tg(l, g, c) = sum_{R_e in group g} e^{2 pi i (j1 n1/m1 + j2 n2/m2)}/de gW(R_e, c)
// with groups of equal n0 mod m0 (about 2 * 10 + 1 of them for a 10^3 R_e grid).
// Stage b (per outer point): g1(k1, c) = sum_g e^{2 pi i j0 n0(g)/m0} Tg(l(k1), g, c):
// k_cache with the groups in the place of R_e and a job per up to 48 points of a
// line, so its products run on the matrix cores too.  A line's 40 points take
// three tiles in one job and Tg is read once; FMAs with the partial sums of all
// groups in registers took 7.7 ms where this takes 5.6 (16 bands, 12 modes, 640 points,
// 21 groups, FP32: 7.1 GB read); what is left is the rotation epilogue.
constexpr int kLineDepth = 4;  // gW rows in flight per thread (16 bytes each)

// NL lines, CPT adjacent columns per thread (one 16-byte load per R_e for
// CPT * sizeof(T2) == 16).  The phase table is (R_e, line): the NL factors of
// one R_e are contiguous, read by the whole workgroup alike.
template <typename T, int NL, int CPT>
__global__ void __launch_bounds__(256) k_cache_line_a(CacheParams p) {
  typedef typename Vec2<T>::type T2;
  typedef T vec __attribute__((ext_vector_type(2 * CPT)));
  constexpr int D = kLineDepth;
  const size_t col0 = (size_t(blockIdx.x) * 256 + threadIdx.x) * CPT;
  const bool ok = col0 < p.N;  // N is a multiple of CPT
  const T2* G = static_cast<const T2*>(p.gW);
  const T2* ph = static_cast<const T2*>(p.phLine);
  T2* out = static_cast<T2*>(p.Tg);
  vec cur[D], nxt[D];
  auto load = [&](vec(&b)[D], int i0) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      const int i = i0 + u;
      if (ok && i < p.nRe) b[u] = *reinterpret_cast<const vec*>(G + size_t(p.reOrder[i]) * p.N + col0);
      else b[u] = vec(T(0));
    }
  };
  load(cur, 0);
  T ar[NL][CPT], ai[NL][CPT];
#pragma unroll
  for (int l = 0; l < NL; ++l)
#pragma unroll
    for (int c = 0; c < CPT; ++c) ar[l][c] = ai[l][c] = T(0);
  for (int i0 = 0; i0 < p.nRe; i0 += D) {
    load(nxt, i0 + D);
#pragma unroll
    for (int u = 0; u < D; ++u) {
      const int i = i0 + u;
      if (i < p.nRe) {
#pragma unroll
        for (int l = 0; l < NL; ++l) {
          const T2 f = ph[size_t(i) * NL + l];
#pragma unroll
          for (int c = 0; c < CPT; ++c) {
            ar[l][c] += f.x * cur[u][2 * c] - f.y * cur[u][2 * c + 1];
            ai[l][c] += f.x * cur[u][2 * c + 1] + f.y * cur[u][2 * c];
          }
        }
        const int g = p.reGroupEnd[i];
        if (g >= 0) {
#pragma unroll
          for (int l = 0; l < NL; ++l) {
            if (ok) {
              vec o;
#pragma unroll
              for (int c = 0; c < CPT; ++c) {
                o[2 * c] = ar[l][c];
                o[2 * c + 1] = ai[l][c];
              }
              *reinterpret_cast<vec*>(out + (size_t(l) * p.nGe + g) * p.N + col0) = o;
            }
#pragma unroll
            for (int c = 0; c < CPT; ++c) ar[l][c] = ai[l][c] = T(0);
          }
        }
      }
    }
#pragma unroll
    for (int u = 0; u < D; ++u) cur[u] = nxt[u];
  }
}

// Stage a for 16 lines on the matrix cores (FP32 data).  Per R_e group g,
// Tg(l, g, c) = sum_{R_e in g} ph(R_e, l) gW(R_e, c) is a complex GEMM with
// M = 16 lines, K = the group's R_e and N = the gW columns.  It runs as real
// products on v_mfma_f32_16x16x4f32, four R_e at a time (groups padded to a
// multiple of 4 with zero entries): lane (n, kq) = (L % 16, L / 16) loads
// gW(R_kq, column n) of each 16-column tile (8 bytes, both components) and
// ph(R_kq, line n), and two K-steps take the x and the y components,
//   Re += a x - b y,   Im += b x + a y      (ph = a + i b, gW = x + i y),
// with A = (a | -b) and (b | a).  D(line 4 kq + i, column n) holds Tg.  A wave
// owns kLineMT tiles of 16 columns and keeps the next block's loads in flight;
// the padded order sits in LDS.  8 bytes of gW per element against 128 FLOPs
// on the matrix cores: bound by HBM.
constexpr int kLineMT = 8;

__global__ void __launch_bounds__(256, 4) k_cache_line_am(CacheParams p) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  extern __shared__ __align__(16) unsigned char smem[];
  int2* sPad = reinterpret_cast<int2*>(smem);  // nRePad
  for (int i = threadIdx.x; i < p.nRePad; i += 256) sPad[i] = p.rePad[i];
  __syncthreads();
  const int lane = threadIdx.x & 63, n = lane & 15, kq = lane >> 4;
  const size_t colw = (size_t(blockIdx.x) * 4 + (threadIdx.x >> 6)) * (16 * kLineMT);
  if (colw >= p.N) return;  // whole waves
  const float2* G = static_cast<const float2*>(p.gW);
  const float2* ph = static_cast<const float2*>(p.phLine);
  float2* out = static_cast<float2*>(p.Tg);
  const int nBlk = p.nRePad / 4;
  auto load = [&](int blk, float2(&v)[kLineMT], float2& f) {
    const int2 e = blk < nBlk ? sPad[4 * blk + kq] : make_int2(-1, -1);
#pragma unroll
    for (int t = 0; t < kLineMT; ++t) {
      const size_t c = colw + 16 * t + n;
      v[t] = (e.x >= 0 && c < p.N) ? G[size_t(e.x) * p.N + c] : make_float2(0.f, 0.f);
    }
    f = e.y >= 0 ? ph[size_t(e.y) * 16 + n] : make_float2(0.f, 0.f);
  };
  f4 re[kLineMT], im[kLineMT];
#pragma unroll
  for (int t = 0; t < kLineMT; ++t) re[t] = im[t] = f4{0.f, 0.f, 0.f, 0.f};
  float2 x[kLineMT], xn[kLineMT], f, fn;
  load(0, x, f);
  for (int b = 0; b < nBlk; ++b) {
    load(b + 1, xn, fn);
#pragma unroll
    for (int t = 0; t < kLineMT; ++t) {
      re[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.x, x[t].x, re[t], 0, 0, 0);
      re[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(-f.y, x[t].y, re[t], 0, 0, 0);
      im[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.y, x[t].x, im[t], 0, 0, 0);
      im[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.x, x[t].y, im[t], 0, 0, 0);
    }
    const int g = p.reBlkEnd[b];
    if (g >= 0) {
#pragma unroll
      for (int t = 0; t < kLineMT; ++t) {
        const size_t c = colw + 16 * t + n;
        if (c < p.N) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            out[(size_t(4 * kq + i) * p.nGe + g) * p.N + c] = make_float2(re[t][i], im[t][i]);
        }
        re[t] = im[t] = f4{0.f, 0.f, 0.f, 0.f};
      }
    }
#pragma unroll
    for (int t = 0; t < kLineMT; ++t) x[t] = xn[t];
    f = fn;
  }
}

template <typename T, int NL>
static void launch_line_a(const CacheParams& p, hipStream_t s) {
  if constexpr (sizeof(T) == 4 && NL == 16) {
    if (p.rePad && p.reBlkEnd && p.nRePad % 4 == 0) {
      const size_t lds = size_t(p.nRePad) * sizeof(int2);
      PHX_REQUIRE(lds <= 160 * 1024, "cacheElPh line: too many R_e for the matrix-core stage");
      PHX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_cache_line_am),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, int(std::max<size_t>(lds, 16))));
      hipLaunchKernelGGL(k_cache_line_am, dim3(ceil_div((long long)p.N, 4 * 16 * kLineMT)), dim3(256), lds, s,
                         p);
      PHX_HIP(hipGetLastError());
      return;
    }
  }
  if constexpr (sizeof(T) == 4) {
    if (p.N % 2 == 0) {
      hipLaunchKernelGGL((k_cache_line_a<T, NL, 2>), dim3(ceil_div((long long)p.N / 2, 256)), dim3(256),
                         0, s, p);
      PHX_HIP(hipGetLastError());
      return;
    }
  }
  {
    hipLaunchKernelGGL((k_cache_line_a<T, NL, 1>), dim3(ceil_div((long long)p.N, 256)), dim3(256), 0, s, p);
  }
  PHX_HIP(hipGetLastError());
}

template <typename T, typename OutT>
void launch_cache_line(const CacheParams& p, hipStream_t s) {
  PHX_REQUIRE(p.nw <= 32, "cacheElPh kernel supports nw <= 32");
  PHX_REQUIRE(p.nGe >= 1 && p.N == size_t(p.nRp) * p.nm * p.nw * p.nw, "cacheElPh line: bad sizes");
  PHX_REQUIRE(p.nLinesB >= 1 && p.nLinesB <= kLinesPerBatch && p.nLinesA == line_count_padded(p.nLinesB),
              "cacheElPh line: 1 to 16 lines per batch");
  PHX_REQUIRE(p.jobs && p.nJobs >= 1 && p.jobTiles >= 1 && p.jobTiles <= kJobTiles,
              "cacheElPh line: bad stage b jobs");
  if (p.nkk <= 0) return;
  switch (p.nLinesA) {
    case 1: launch_line_a<T, 1>(p, s); break;
    case 2: launch_line_a<T, 2>(p, s); break;
    case 3: launch_line_a<T, 3>(p, s); break;
    case 4: launch_line_a<T, 4>(p, s); break;
    case 6: launch_line_a<T, 6>(p, s); break;
    case 8: launch_line_a<T, 8>(p, s); break;
    case 12: launch_line_a<T, 12>(p, s); break;
    default: launch_line_a<T, 16>(p, s); break;
  }
  launch_cache_gemm<T, OutT>(p, p.jobTiles, p.nJobs, s);  // stage b
}
template void launch_cache_line<double, double>(const CacheParams&, hipStream_t);
template void launch_cache_line<float, float>(const CacheParams&, hipStream_t);

// FP64 -> FP32 copy of the coupling tensor (the reduced-precision GEMMs read it).
__global__ void k_to_float(const double* __restrict__ a, float* __restrict__ b, size_t n) {
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x)
    b[i] = float(a[i]);
}
void launch_to_float(const double* a, float* b, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_to_float, dim3(8192), dim3(256), 0, s, a, b, n);
  PHX_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ coupling
// (coupling_kernel.hpp, instantiated in coupling_f64.hip and coupling_f32.hip)

// ------------------------------------------------------------------ collect

// One workgroup per (k1, b1): 256 threads stride over the partial slots of the
// panels of b1's degenerate group, then a fixed-order tree sum (deterministic).
__global__ void __launch_bounds__(256) k_collect(CollectParams p) {
  __shared__ double red[4][kCMax];
  const int kk = blockIdx.x, b1 = blockIdx.y;
  if (kk >= p.nkk || b1 >= p.kkNb1[kk]) return;  // uniform per workgroup
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int pan = p.kkPanelBase[kk] + b1;
  const int gs = p.panelGStart[pan], gz = p.panelGSize[pan];
  double sum[kCMax] = {0., 0., 0., 0.};
  const int n = gz * p.nMtiles;
  for (int i = t; i < n; i += 256) {
    const int j = i / p.nMtiles, mt = i - j * p.nMtiles;
    const int src = p.kkPanelBase[kk] + gs + j;
    const double2* q = reinterpret_cast<const double2*>(
        p.partial + (size_t(src) * p.nMtiles + mt) * kGMax * kCMax + (b1 - gs) * kCMax);
    const double2 v0 = q[0], v1 = q[1];
    sum[0] += v0.x;
    sum[1] += v0.y;
    sum[2] += v1.x;
    sum[3] += v1.y;
  }
#pragma unroll
  for (int c = 0; c < kCMax; ++c) {
    double v = sum[c];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    if (lane == 0) red[wave][c] = v;
  }
  __syncthreads();
  if (t < p.nCalc)
    p.linewidth[size_t(t) * p.numStates + p.kkStateOff[kk] + b1] +=
        ((red[0][t] + red[1][t]) + (red[2][t] + red[3][t]));
}

void launch_collect(const CollectParams& p, hipStream_t s) {
  if (p.nkk <= 0) return;
  hipLaunchKernelGGL(k_collect, dim3(p.nkk, p.nb1Max), dim3(256), 0, s, p);
  PHX_HIP(hipGetLastError());
}

}  // namespace phx
