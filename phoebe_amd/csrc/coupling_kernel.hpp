// Coupling kernels for one batch of outer points k1 (panels = (k1, b1) pairs):
//
//  * k_coupling  : direct R_ph transform, g3(row, c) = sum_Rp e^{ik2.Rp} C(Rp, c)
//                  (or e^{iq.Rp} for explicit q) on v_mfma_{f64,f32}_16x16x4,
//                  followed by the shared epilogue;
//  * k_sep_*     : the same g3 for k2 on the Gamma-centred mesh as three short
//                  lattice-direction transforms e^{ik2.Rp} = prod_d w_d^{j_d n_d}
//                  (w_d = e^{2 pi i / m_d}, n = integer coordinates of Rp folded
//                  mod m), the last one fused with the shared epilogue.
//
// Shared epilogue (per 16 rows, g3(nu, w2) of each row in LDS):
//   g'(nu, b2)  = sum_w2 conj(U2(w2, b2)) g3(nu, w2)    (interaction_elph.cpp:393-402)
//   g(nu2, b2)  = sum_nu e3(nu, nu2) g'(nu, b2)         (interaction_elph.cpp:381-390)
// i.e. the reference's two rotations applied in the cheaper order (the electron
// rotation first shrinks w2 -> b2), then |g|^2 and either a store in the
// getCouplingSquared layout or symmetrizeCoupling along b2 and nu plus the
// Gaussian-delta weights of el_scattering.cpp:277-380 into per-workgroup partials.
//
// Instantiated per precision of the transforms in coupling_f64.hip / coupling_f32.hip.
#pragma once

#include <algorithm>
#include <type_traits>

#include "coupling_tiling.hpp"
#include "elph_params.hpp"
#include "last_stage.hpp"
#include "phx_common.hpp"

namespace phx {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));

constexpr int kNmMax = 36;

struct CoupParams {
  // direct transform operands
  const void* A; size_t lda;              // (R_p rounded up to quads, rows): e^{ik2.Rp} complex, zero beyond R_p; row length lda
  const void* B; size_t panelStride; int ldb;  // panels (R_p, col) complex, ldb reals per R_p
  int M, nRp, nm, nw, nPanels, nMtiles;
  const int* panelKK;
  const int* panelB1;
  // rows
  const double2* U2pool; const int* rowU2off; const int* rowNb2;
  // phonons
  const double2* E3pool; const double* Wpool;
  int qmode;                              // 0: e3 index = rowE3[row]; 1: mesh difference
  const int* rowE3; const int* rowMesh; const int* kkMesh; int m0, m1, m2;
  // store mode (calcCouplingSquared): out(q)(b1 + nb1 (b2 + nb2 nu))
  double* out; const long long* rowOutOff; const int* kkNb1;
  // several outer points per launch with rows of their own: added per kk to rowU2off and out
  long long rowKKStride, outKKStride;
  // reduce mode
  const double* e2pool; const int* rowStateOff;
  const double* e1pool; const int* kkStateOff;
  const int* panelGStart; const int* panelGSize;
  const double* fermi; int numStates;
  const double* bose;                     // (q, nu, calc)
  int nCalc; double invSigma, deltaPref, norm, cutoff;
  int gsizeMax;                           // largest panelGSize of the launch (0: unknown, kGMax)
  double* partial;                        // (L = panel*nMtiles + mtile, kGMax, kCMax)
  int nb2max;
  // separable mesh transform
  const int* meshToRow;                   // full mesh index -> row (active point) or -1
  const void* T2; size_t t2PanelStride;   // (panel, f0 group, jy, jz, col) complex
  int nG0; const int* g0val;              // folded x coordinate of each group
  const double2* tw0;                     // e^{2 pi i t / m0}, t < m0
  int rowLo, rowHi;                       // rows (active indices) taken by the mesh transform
  double screen;                          // energy screen in units of sigma (0: off)
  double* screenOf;                       // per outer state: screen width (sigma) of the panel whose b1 group
                                          // starts there (k_sep_xmin); null: `screen` for every panel
  double* xminPart;                       // (panel, kXminBlocks) closest approach to resonance, energy units
  const double* qWlo; const double* qWhi; // per q: lowest / highest omega >= cutoff
  const double2* rowE2range;              // per row: (lowest, highest) band energy
  // learned screen (k_sep_xm): per (panel, yz) slot masks
  int bf16x3;                             // x-stage GEMMs in split-BF16x3 (FP32 data)
  const unsigned char* slotOn;            // compute only slots with slotOn != 0 (null: all)
  int slotZero;                           // off slots: 1 = write zero partials, 0 = leave untouched
  const int* gate;                        // run only when *gate != 0 (null: always)
  unsigned long long* keptRows;           // rows computed by the last stage are added here (null: off)
  // precomputed row lists of the last stage (m0 <= 64)
  unsigned long long* keepMask;           // per slot: bit jx set = row jx kept (null: screen in k_sep_xm)
  const int4* meshRow;                    // per mesh point: (row, nb2, u2off, stateOff), row -1 if inactive
  // adaptive Gaussian smearing: width from the group velocities of the two states
  int adaptive;                           // 0: fixed Gaussian (invSigma, deltaPref)
  const double* stateV;                   // numStates x 3 group velocities
  double qT[9];                           // reciprocal cell, row i divided by mesh(i), row-major
  double minWidth;                        // smallest width (0.1 meV)
  // degenerate phonon modes: per q and mode, first mode of its group | group size << 8
  const int* qModeGrp;
  // separable transform: phonon eigenvectors (q, nu, nu2) in the transform's precision
  const void* E3T;
  // polar term (direct transform epilogue): per e3 index (row of the per-call
  // API, folded q of the builder) nm complex polarCorrectionPart1 values, zero
  // where the reference skips the term; U1 of the outer point: U1pool +
  // U1off[kk], (nw, nb1) column-major.  polarX null: no polar term.
  const double2* polarX;
  const double2* U1pool;
  const int* U1off;
  // split last stage (k_sep_yx or k_sep_xg, then k_sep_ep2): g3 rows of the chunk, (slot, jx, col) complex T
  void* G3;
  unsigned long long* keptBands;          // k_sep_ep2: sum of nb2 over the rows it computed (null: off)
  int stage;                              // kernels of the last stage (LastStage)
  unsigned long long* keptSlots;          // k_sep_xg: slots (panel, yz line) it computed (null: off)
};

template <typename T> struct Vec2;
template <> struct Vec2<double> { typedef double2 type; };
template <> struct Vec2<float> { typedef float2 type; };

// Energy-screen width, in units of sigma, of the panel whose b1 group starts
// at outer state is1 (see k_sep_xmin).
__device__ inline double screen_width(const CoupParams& p, int is1) {
  return p.screenOf ? p.screenOf[is1] : p.screen;
}

__device__ inline double gaussian_delta(double energy, double invW, double pref) {
  // GaussianDeltaFunction::getSmearing, delta_function.cpp:40-45
  double x = energy * invW;
  if (x > 6.) return 0.;
  return pref * exp(-x * x);
}

// AdaptiveGaussianDeltaFunction::getSmearing (delta_function.cpp:66-97) with
// v = v(state 1) - v(state 2) (el_scattering.cpp:291-295): width
// sqrt(sum_i (qT_i . v)^2 / 6), at least minWidth; cut at 2 widths and
// renormalized by erf(2).
struct AdaptiveWidth {
  double sigma;  // 0: delta is zero; < 0: zero velocity difference
};
__device__ inline AdaptiveWidth adaptive_width(const CoupParams& p, int is1, int is2) {
  const double v0 = p.stateV[3 * is1] - p.stateV[3 * is2];
  const double v1 = p.stateV[3 * is1 + 1] - p.stateV[3 * is2 + 1];
  const double v2 = p.stateV[3 * is1 + 2] - p.stateV[3 * is2 + 2];
  AdaptiveWidth w;
  if (v0 == 0. && v1 == 0. && v2 == 0.) {
    w.sigma = -1.;
    return w;
  }
  double s = 0.;
  for (int i = 0; i < 3; ++i) {
    const double d = p.qT[3 * i] * v0 + p.qT[3 * i + 1] * v1 + p.qT[3 * i + 2] * v2;
    s += d * d;
  }
  s = sqrt(s / 6.);
  if (s != 0. && s < p.minWidth) s = p.minWidth;
  w.sigma = s;
  return w;
}
__device__ inline double adaptive_delta(double energy, AdaptiveWidth w) {
  if (w.sigma < 0.) return energy == 0. ? 1. : 0.;
  if (w.sigma == 0.) return 0.;
  if (fabs(energy) > 2. * w.sigma) return 0.;
  const double x = energy / w.sigma;
  if (x > 6.) return 0.;
  return exp(-x * x) / 1.7724538509055160273 / w.sigma / 0.9953222650189527;
}

// FP64 / FP32 main loop on v_mfma_*_16x16x4: A lane l holds A[l%16][l/16], B lane l holds
// B[l/16][l%16].  Accumulator i of lane l is D[row(l/16, i)][l%16] with
// row = l/16 + 4i for f64 and 4(l/16) + i for f32 (measured on gfx950).
template <typename T> struct Mfma4;
template <> struct Mfma4<double> {
  typedef d4_t acc_t;
  __device__ static acc_t mac(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static int row(int lk, int i) { return lk + 4 * i; }
};
template <> struct Mfma4<float> {
  typedef f4_t acc_t;
  __device__ static acc_t mac(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static int row(int lk, int i) { return 4 * lk + i; }
};

// Electron rotation of the modes nuLo .. nuHi-1 for the 16 rows whose g3
// blocks are in LDS (row r at g3 + r*PWp, (re, im) of column (nu, w2) at
// 2((nu - nuLo)*nw + w2)) into g'(nu, b2) in scratch.  Thread t serves row t/16.
template <typename T>
__device__ void epilogue16_u2(const CoupParams& p, const T* g3, int PWp, unsigned char* scratch,
                              int myRow, int nuLo, int nuHi) {
  const int t = threadIdx.x, r = t >> 4, sub = t & 15;
  const int nw = p.nw;
  const int stride = p.nm * p.nb2max;
  double2* gp = reinterpret_cast<double2*>(scratch) + size_t(r) * stride;
  const bool valid = myRow >= 0;
  const int nb2 = valid ? p.rowNb2[myRow] : 0;
  const T* g = g3 + size_t(r) * PWp;
  const double2* U2 = p.U2pool + (valid ? p.rowU2off[myRow] : 0);
  for (int o = sub; o < (nuHi - nuLo) * nb2; o += 16) {
    const int nl = o / nb2, b2 = o % nb2;
    double2 s = make_double2(0., 0.);
#pragma unroll 8
    for (int w2 = 0; w2 < nw; ++w2) {
      const double2 u = U2[w2 + nw * b2];
      const double xr = double(g[2 * (nl * nw + w2)]), xi = double(g[2 * (nl * nw + w2) + 1]);
      s.x += u.x * xr + u.y * xi;
      s.y += u.x * xi - u.y * xr;
    }
    gp[(nuLo + nl) * nb2 + b2] = s;
  }
}

// Rest of the epilogue once g'(nu, b2) of every mode is in scratch: phonon
// rotation, |g|^2, then the store or the symmetrization and the weights.
// Must be called by all 256 threads.  stage (null: none): LDS of 16 (nm +
// nb2max) doubles for the rows' frequencies and band energies, which the search
// for degenerate groups would else read from memory one after the other.
template <bool REDUCE>
__device__ void epilogue16_tail(const CoupParams& p, unsigned char* scratch, double* stage, int panel, int kk, int b1p,
                                int myRow, int myIq, double (&part)[kGMax][kCMax]) {
  const int t = threadIdx.x, r = t >> 4, sub = t & 15;
  const int nm = p.nm;
  const int stride = nm * p.nb2max;
  double2* gp = reinterpret_cast<double2*>(scratch) + size_t(r) * stride;
  double* gs = reinterpret_cast<double*>(reinterpret_cast<double2*>(scratch) + size_t(16) * stride) +
               size_t(r) * stride;
  const bool valid = myRow >= 0;
  const int nb2 = valid ? p.rowNb2[myRow] : 0;
  const double2* e3 = p.E3pool + size_t(myIq) * nm * nm;
  const bool polar = p.polarX != nullptr && valid;
  const double* const w3g = p.Wpool + size_t(myIq) * nm;
  const double* const e2g = REDUCE ? p.e2pool + (valid ? p.rowStateOff[myRow] : 0) : nullptr;  // no states in store mode
  double* const w3s = stage ? stage + r * nm : nullptr;
  double* const e2s = stage ? stage + 16 * nm + r * p.nb2max : nullptr;
  if (REDUCE && stage && valid) {
    for (int i = sub; i < nm; i += 16) w3s[i] = w3g[i];
    for (int i = sub; i < nb2; i += 16) e2s[i] = e2g[i];
  }
  for (int o = sub; o < nm * nb2; o += 16) {
    const int nu2 = o / nb2, b2 = o % nb2;
    double2 s = make_double2(0., 0.);
#pragma unroll 6
    for (int nu = 0; nu < nm; ++nu) {
      const double2 e = e3[nu + nm * nu2], x = gp[nu * nb2 + b2];
      s.x += x.x * e.x - x.y * e.y;
      s.y += x.x * e.y + x.y * e.x;
    }
    if (polar) {
      // gFinal += x(nu2) <U2(b2)|U1(b1)> (interaction_elph.cpp:406-413 with
      // polarCorrectionPart2, :205-227)
      const double2* u1 = p.U1pool + p.U1off[kk] + size_t(p.nw) * b1p;
      const double2* u2 = p.U2pool + p.rowU2off[myRow] + size_t(p.nw) * b2;
      double2 ov = make_double2(0., 0.);
      for (int w = 0; w < p.nw; ++w) {
        const double2 a = u2[w], b = u1[w];
        ov.x += a.x * b.x + a.y * b.y;
        ov.y += a.x * b.y - a.y * b.x;
      }
      const double2 x = p.polarX[size_t(myIq) * nm + nu2];
      s.x += x.x * ov.x - x.y * ov.y;
      s.y += x.x * ov.y + x.y * ov.x;
    }
    const double v = s.x * s.x + s.y * s.y;
    if (REDUCE) {
      gs[nu2 * nb2 + b2] = v;
    } else {
      const int nb1 = p.kkNb1[kk];
      p.out[p.rowOutOff[myRow] + b1p + size_t(nb1) * (b2 + size_t(nb2) * nu2)] = v;
    }
  }
  if (!REDUCE) return;
  __syncthreads();

  auto w3 = [&](int i) { return stage ? w3s[i] : w3g[i]; };
  auto e2 = [&](int i) { return stage ? e2s[i] : e2g[i]; };
  // symmetrizeCoupling (scattering.cpp:1209-1318) along b2, then nu
  for (int nu = sub; nu < nm && valid; nu += 16) {
    for (int b = 0; b < nb2; ++b) {
      int deg = 0;
      for (int i = b; i < nb2; ++i) {
        if (fabs(e2(b) - e2(i)) < 1.0e-6) deg++;
        else break;
      }
      if (deg > 1) {
        double s = 0.;
        for (int i = 0; i < deg; ++i) s += gs[nu * nb2 + b + i] / double(float(deg));
        for (int i = 0; i < deg; ++i) gs[nu * nb2 + b + i] = s;
      }
      b += deg - 1;
    }
  }
  __syncthreads();
  for (int b2 = sub; b2 < nb2; b2 += 16) {
    for (int nu = 0; nu < nm; ++nu) {
      int deg = 0;
      for (int i = nu; i < nm; ++i) {
        if (fabs(w3(nu) - w3(i)) < 1.0e-6) deg++;
        else break;
      }
      if (deg > 1) {
        double s = 0.;
        for (int i = 0; i < deg; ++i) s += gs[(nu + i) * nb2 + b2] / double(float(deg));
        for (int i = 0; i < deg; ++i) gs[(nu + i) * nb2 + b2] = s;
      }
      nu += deg - 1;
    }
  }
  __syncthreads();

  // Gaussian-delta weights (el_scattering.cpp:277-380, switchCase 2)
  const int gstart = p.panelGStart[panel], gsize = p.panelGSize[panel];
  const double* e1 = p.e1pool + p.kkStateOff[kk];
  const int nCalc = p.nCalc;
  const double inv_g = 1. / double(float(gsize));
  for (int o = sub; o < nm * nb2; o += 16) {
    const int nu = o / nb2, b2 = o % nb2;
    const double en3 = w3(nu);
    if (en3 < p.cutoff) continue;
    const double cpl = gs[nu * nb2 + b2] * inv_g;
    const double en2 = e2(b2);
    const int is2 = p.rowStateOff[myRow] + b2;
#pragma unroll
    for (int gi = 0; gi < kGMax; ++gi) {
      if (gi >= gsize) break;
      const double en1 = e1[gstart + gi];
      double d1, d2;
      if (p.adaptive) {
        const AdaptiveWidth aw = adaptive_width(p, p.kkStateOff[kk] + gstart + gi, is2);
        d1 = adaptive_delta(en1 - en2 + en3, aw);
        d2 = adaptive_delta(en1 - en2 - en3, aw);
      } else {
        d1 = gaussian_delta(en1 - en2 + en3, p.invSigma, p.deltaPref);
        d2 = gaussian_delta(en1 - en2 - en3, p.invSigma, p.deltaPref);
      }
      if (d1 <= 0. && d2 <= 0.) continue;
#pragma unroll
      for (int c = 0; c < kCMax; ++c) {
        if (c >= nCalc) break;
        const double f2 = p.fermi[size_t(c) * p.numStates + is2];
        const double n3 = p.bose[(size_t(myIq) * nm + nu) * nCalc + c];
        part[gi][c] += cpl * ((f2 + n3) * d1 + (1. - f2 + n3) * d2) * p.norm / en3 * 3.14159265358979323846;
      }
    }
  }
}

// Block reduction of the per-thread partial linewidths into partial[L]
// (CM calculations and GM group members held per thread; the slots beyond
// them are written as zero).
template <int CM, int GM = kGMax, int NWV = 4>
__device__ inline void reduce_partials(const CoupParams& p, int L, unsigned char* smem,
                                       double (&part)[GM][CM]) {
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  double* red = reinterpret_cast<double*>(smem);
  __syncthreads();
#pragma unroll
  for (int gi = 0; gi < GM; ++gi)
#pragma unroll
    for (int c = 0; c < CM; ++c) {
      double v = part[gi][c];
      for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
      if (lane == 0) red[(gi * kCMax + c) * NWV + wave] = v;
    }
  __syncthreads();
  if (t < kGMax * kCMax) {
    const int c = t % kCMax, gi = t / kCMax;
    double v = 0.;
    if (c < CM && gi < GM)
#pragma unroll
      for (int w = 0; w < NWV; ++w) v += red[t * NWV + w];
    p.partial[size_t(L) * kGMax * kCMax + t] = v;
  }
}

// ------------------------------------------------------------------ direct transform
// (coupling_direct.hpp, instantiated in coupling_direct_f64.hip and coupling_direct_f32.hip)

static_assert(kCoupReduceLds == size_t(kGMax) * kCMax * 4 * sizeof(double), "LDS of reduce_partials");
template <typename T>
void launch_coupling(const CoupParams& p, bool reduce, hipStream_t s);

// ------------------------------------------------------------------ separable transform
// Integer layout of the R_ph set folded on the mesh:
//   lines  = distinct (f0, f1), entries (f2, Rp)          (stage z)
//   groups = distinct f0,       entries (f1, line)        (stage y)
struct SepParams {
  const void* B; size_t panelStride; int ldb;   // panels: C(Rp, col), ldb reals per Rp
  int ncol, nPanels, mx, my, mz;
  int modeFast;                                 // nm: columns of T1 / T2 / g3 as (w2, nu); 0: as the panels, (nu, w2)
  int nLines; const int* lineStart; const int* lineF2; const int* lineRp;
  const double2* twz;                           // e^{2 pi i t / mz}
  void* T1; size_t t1PanelStride;               // (panel, line, jz, col)
  int nG0;
  // the groups' entries in quads (the last one padded), the groups dealt to four waves: wave w sums
  // quads waveQ[w] .. waveQ[w + 1] - 1; entry (line, f1), line -1 = padding; quadEnd: group that ends
  // with the quad, or -1
  int nQuads; int waveQ[5]; const int2* quadEnt; const int* quadEnd;
  const double2* twy;                           // e^{2 pi i t / my}
  void* T2; size_t t2PanelStride;               // (panel, group, jy, jz, col)
};

// Register-blocked short transform of k_sep_z:
// out(j, c) = sum_e W(e, j) X(e, c) for j < m, c < ncol, X (the data's
// precision, converted to FP64 on reading) and W in LDS.
// Thread (wave w, lane l) takes the columns c = l, l + 64, ... and the rows
// j = w + 4 i, kSepJB of them at once, so one LDS read of X(e, c) serves
// kSepJB rows and W(e, j) is the same for the whole wave (a broadcast); no
// integer division.  Every output sums its terms in ascending e, as a plain
// loop over the outputs would.
constexpr int kSepJB = 10;
template <typename T, typename Store>
__device__ __forceinline__ void sep_short_transform(const typename Vec2<T>::type* X, const double2* W, int ne,
                                                    int m, int ncol, Store store) {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
  for (int c = l; c < ncol; c += 64) {
    for (int j0 = w; j0 < m; j0 += 4 * kSepJB) {
      double2 acc[kSepJB];
#pragma unroll
      for (int i = 0; i < kSepJB; ++i) acc[i] = make_double2(0., 0.);
      for (int e = 0; e < ne; ++e) {
        const typename Vec2<T>::type xv = X[e * ncol + c];
        const double2 x = make_double2(double(xv.x), double(xv.y));
        const double2* we = W + e * m;
#pragma unroll
        for (int i = 0; i < kSepJB; ++i) {
          const int j = j0 + 4 * i;
          if (j < m) {
            const double2 ww = we[j];
            acc[i].x += ww.x * x.x - ww.y * x.y;
            acc[i].y += ww.x * x.y + ww.y * x.x;
          }
        }
      }
#pragma unroll
      for (int i = 0; i < kSepJB; ++i)
        if (j0 + 4 * i < m) store(j0 + 4 * i, c, acc[i]);
    }
  }
}

// Entries of a short transform into LDS: X(e, c) = row(e)[c] for e < ne,
// c < ncol (the data's precision), and the twiddles W(e, j) = tw[(j f(e)) mod m],
// j < m.  The rows' offsets and the f(e) are staged first (off, fe: ne ints
// each); every thread then keeps up to 8 row loads in flight before its LDS
// stores, so a workgroup waits about one memory latency, not one per entry.
// nm > 0: column c = nu (ncol / nm) + w2 goes to w2 nm + nu.
template <typename T2v, typename Meta>
__device__ __forceinline__ void sep_stage_entries(const T2v* base, T2v* X, double2* W, int* off, int* fe, int ne,
                                                  int ncol, int m, int nm, const double2* tw, Meta meta) {
  const int t = threadIdx.x, bs = blockDim.x;
  for (int e = t; e < ne; e += bs) meta(e, off[e], fe[e]);
  __syncthreads();
  const int n = ne * ncol;
  for (int i0 = t; i0 < n; i0 += 8 * bs) {
    T2v v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = i0 + bs * u;
      if (i < n) {
        const int e = i / ncol;
        v[u] = base[size_t(off[e]) + (i - e * ncol)];
      }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = i0 + bs * u;
      if (i < n) {
        int d = i;
        if (nm > 0) {
          const int e = i / ncol, c = i - e * ncol, nw = ncol / nm, nu = c / nw;
          d = e * ncol + (c - nu * nw) * nm + nu;
        }
        X[d] = v[u];
      }
    }
  }
  for (int i = t; i < ne * m; i += bs) {
    const int e = i / m, j = i - e * m;
    W[i] = tw[(j * fe[e]) % m];
  }
  __syncthreads();
}

// LDS of k_sep_z for ne entries: X (ne x ncol in the data's
// precision), W (ne x m complex FP64), the entries' row offsets and factors.
inline size_t sep_stage_lds_bytes(int elem, int ne, int ncol, int m) {
  const size_t x = (size_t(ne) * ncol * 2 * elem + 15) / 16 * 16;
  return x + size_t(ne) * m * sizeof(double2) + size_t(ne) * 2 * sizeof(int);
}

// T1(line, jz, c) = sum_{(f2, Rp) in line} w_z^{jz f2} C(Rp, c).  The line's
// entries and their twiddles w_z^{jz f2} (an entries x mz table) sit in LDS.
// The panels' columns are (nu, w2); with modeFast the staging turns them into
// (w2, nu) for the split last stage, whose epilogue reads them with the modes in
// neighbouring lanes.
template <typename T>
__global__ void __launch_bounds__(256) k_sep_z(SepParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef typename Vec2<T>::type T2v;
  const int line = blockIdx.x, panel = blockIdx.y;
  const int e0 = p.lineStart[line], ne = p.lineStart[line + 1] - e0;
  const int ncol = p.ncol, mz = p.mz;
  T2v* X = reinterpret_cast<T2v*>(smem);  // (entries, ncol)
  double2* W = reinterpret_cast<double2*>(smem + (size_t(ne) * ncol * sizeof(T2v) + 15) / 16 * 16);  // (entries, mz)
  int* off = reinterpret_cast<int*>(W + size_t(ne) * mz);
  int* fe = off + ne;
  const T2v* B = reinterpret_cast<const T2v*>(static_cast<const T*>(p.B) + size_t(panel) * p.panelStride);
  sep_stage_entries(B, X, W, off, fe, ne, ncol, mz, p.modeFast, p.twz, [&](int e, int& o, int& f) {
    o = p.lineRp[e0 + e] * (p.ldb / 2);
    f = p.lineF2[e0 + e];
  });
  T2v* out = reinterpret_cast<T2v*>(static_cast<T*>(p.T1) + size_t(panel) * p.t1PanelStride) +
             size_t(line) * mz * ncol;
  sep_short_transform<T>(X, W, ne, mz, ncol, [&](int jz, int c, double2 v) {
    out[size_t(jz) * ncol + c] = T2v{T(v.x), T(v.y)};
  });
}

// ------------------------------------------------------------------ y-stage on the matrix cores
// T2(g, jy, c) = sum_{(f1, line) in group g} w_y^{jy f1} T1(line, jz, c) for 16
// y coordinates and 16 columns at once on v_mfma_f64_16x16x4, N = columns, K = a
// quad of the group's entries.  The coordinates go in pairs jy, my - jy, whose
// twiddles are conjugate: with C = sum cos x and S = sum sin x over the entries,
// T2(jy) = (Re C - Im S, Im C + Re S) and T2(my - jy) = (Re C + Im S, Im C - Re S).
// Rows 0..7 of M are the cosines of eight pairs and rows 8..15 their sines, so that
// a pair's C and S are registers of the same lane, and a quad takes two products
// (x's real and imaginary parts) where one coordinate per row took four.  The pair
// of jy = 0 has no sines; for even my its S rows hold w^{f1 my / 2} = (-1)^f1, and
// S is T2(my / 2).  The groups are dealt to the four waves by the host (waveQ), so
// a group's sum stays in one wave's registers, in ascending order of its
// entries; T1 goes from L2 straight to registers, four quads ahead.  FP64 sums
// of the data's precision, rounded once on storing.
// Shared by k_sep_y and k_sep_yx, which so give the same T2 bit for bit.
struct SepYShared {
  double* tw;  // my: cos(2 pi t / my), then my: sin
  int2* ent;   // 4 nQuads: (T1 row at jz: offset of its first column, or -1: padding; f1)
  int* end;    // nQuads: group that ends with the quad, or -1
};
__device__ __forceinline__ SepYShared sep_y_stage(const SepParams& p, unsigned char* smem, int jz) {
  SepYShared s;
  s.tw = reinterpret_cast<double*>(smem);
  s.ent = reinterpret_cast<int2*>(s.tw + 2 * p.my);
  s.end = reinterpret_cast<int*>(s.ent + 4 * p.nQuads);
  for (int i = threadIdx.x; i < p.my; i += 256) {
    const double2 w = p.twy[i];
    s.tw[i] = w.x;
    s.tw[p.my + i] = w.y;
  }
  for (int i = threadIdx.x; i < 4 * p.nQuads; i += 256) {
    const int2 e = p.quadEnt[i];
    s.ent[i] = make_int2(e.x < 0 ? -1 : (e.x * p.mz + jz) * p.ncol, e.y);
  }
  for (int i = threadIdx.x; i < p.nQuads; i += 256) s.end[i] = p.quadEnd[i];
  return s;
}
// The pairs of a y mesh, and the coordinate of a tile's place jj (pairs r0 .. r0 + 7:
// places 0..7 their first coordinates, 8..15 their second ones), or -1.
__host__ __device__ inline int sep_y_pairs(int my) { return (my + 1) / 2; }
__device__ __forceinline__ int sep_y_coord(int my, int r0, int jj) {
  const int r = r0 + (jj & 7);
  if (r >= sep_y_pairs(my)) return -1;
  if (jj < 8) return r;
  return r > 0 ? my - r : my % 2 == 0 ? my / 2 : -1;
}
// store(g, jj, re, im): column min(col0 + lane % 16, ncol - 1) of place jj's y coordinate
// (for places without one, of no meaning)
template <typename T, typename Store>
__device__ __forceinline__ void sep_y_tile(const SepParams& p, const SepYShared& s,
                                           const typename Vec2<T>::type* T1, int col0, int r0, Store store) {
  typedef typename Vec2<T>::type T2v;
  constexpr int NQ = 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, lr = lane & 15,
            lg = lane >> 4;
  const int q0 = p.waveQ[wave], q1 = p.waveQ[wave + 1];
  if (q0 == q1) return;
  const T2v* src = T1 + min(col0 + lr, p.ncol - 1);
  // the lane's twiddles: cosines of coordinate r0 + lr, or sines of r0 + lr - 8
  const bool half = r0 == 0 && lr == 8;  // S row of jy = 0: cosines of my / 2
  const int jy = half ? p.my / 2 : r0 + (lr & 7);
  const double* tw = s.tw + (lr < 8 || half ? 0 : p.my);
  const float invMy = 1.f / float(p.my);
  T2v x[NQ], xn[NQ];
  int2 e[NQ], en[NQ];
  auto load = [&](T2v(&v)[NQ], int2(&w)[NQ], int q) {
#pragma unroll
    for (int u = 0; u < NQ; ++u) {
      w[u] = s.ent[4 * min(q + u, q1 - 1) + lg];
      v[u] = src[max(w[u].x, 0)];
    }
  };
  d4_t re = {0., 0., 0., 0.}, im = {0., 0., 0., 0.};
  load(x, e, q0);
  for (int q = q0; q < q1; q += NQ) {
    load(xn, en, q + NQ);
#pragma unroll
    for (int u = 0; u < NQ; ++u) {
      if (q + u < q1) {
        // (jy f1) mod my: the quotient through a float is off by at most one
        const int n = jy * e[u].y;
        int r = n - int(float(n) * invMy) * p.my;
        r += r < 0 ? p.my : 0;
        r -= r >= p.my ? p.my : 0;
        const bool on = e[u].x >= 0;
        const double w = tw[r];
        re = Mfma4<double>::mac(w, on ? double(x[u].x) : 0., re);
        im = Mfma4<double>::mac(w, on ? double(x[u].y) : 0., im);
        const int g = __builtin_amdgcn_readfirstlane(s.end[q + u]);
        if (g >= 0) {
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const int r = Mfma4<double>::row(lg, i);  // < 8; its sines are row(lg, i + 2) = r + 8
            const bool zero = r0 + r == 0;
            store(g, r, zero ? re[i] : re[i] - im[i + 2], zero ? im[i] : im[i] + re[i + 2]);
            store(g, r + 8, zero ? re[i + 2] : re[i] + im[i + 2], zero ? im[i + 2] : im[i] - re[i + 2]);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) re[i] = im[i] = 0.;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < NQ; ++u) {
      x[u] = xn[u];
      e[u] = en[u];
    }
  }
}

// The y-stage alone, T2 to device memory.  Grid (blocks of 16 columns, jz, panels).
template <typename T>
__global__ void __launch_bounds__(256) k_sep_y(SepParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef typename Vec2<T>::type T2v;
  const int jz = blockIdx.y, panel = blockIdx.z, col0 = blockIdx.x * 16;
  const int c = col0 + (threadIdx.x & 15);
  const SepYShared s = sep_y_stage(p, smem, jz);
  __syncthreads();
  const T2v* T1 = reinterpret_cast<const T2v*>(static_cast<const T*>(p.T1) + size_t(panel) * p.t1PanelStride);
  T2v* out = reinterpret_cast<T2v*>(static_cast<T*>(p.T2) + size_t(panel) * p.t2PanelStride) + c;
  for (int r0 = 0; r0 < sep_y_pairs(p.my); r0 += 8)
    sep_y_tile<T>(p, s, T1, col0, r0, [&](int g, int jj, double re, double im) {
      const int jy = sep_y_coord(p.my, r0, jj);
      if (jy >= 0 && c < p.ncol) out[((size_t(g) * p.my + jy) * p.mz + jz) * p.ncol] = T2v{T(re), T(im)};
    });
}

// Last stage + epilogue for one (jy, jz) line of mesh points and one panel.
//
//  1. rows of the line: active point, q index, and (screen > 0) the energy
//     screen: a row is kept only if some e1 of the panel's degenerate group,
//     band e2 of the row and mode omega >= cutoff at q give
//     |e1 - e2 +- omega| < screen * sigma (an interval test on the band and
//     mode ranges, so no contributing row is dropped; every skipped term has
//     all its Gaussians below exp(-screen^2) of their peak);
//  2. surviving rows, 8 per pass: g3(jx; c) = sum_groups w_x^{jx f0} T2(group, jy, jz, c);
//  3. epilogue with 32 threads per row: thread nu2 owns the column e3(., nu2) (prefetched),
//     g'(nu, b2) via U2 staged in LDS, g(nu2, b2) and |g|^2 for all b2 in registers,
//     symmetrization along b2 in registers and along nu through LDS (only when the
//     modes at q are degenerate), Gaussian weights.
constexpr int kSepRows = 8;   // rows per pass
constexpr int kSepNb2 = 8;    // largest band count of an inner point on this path
constexpr int kSepNm = 32;    // largest mode count on this path

struct SepXShared {            // per-row data staged in LDS
  int row, iq, nb2, u2off, soff;
};

template <typename T, bool REDUCE, int NMX, int CM>
__global__ void __launch_bounds__(256, 2) k_sep_x(CoupParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef typename Vec2<T>::type T2v;
  const int nLinesYZ = p.m1 * p.m2;
  const int nTilesTot = p.nPanels * nLinesYZ;
  const int bid = blockIdx.x;
  const int perXcd = gridDim.x / 8;
  const int L = (bid % 8) * perXcd + bid / 8;
  if (L >= nTilesTot) return;
  const int panel = L / nLinesYZ, yz = L % nLinesYZ;
  const int jy = yz % p.m1, jz = yz / p.m1;
  const int t = threadIdx.x;
  const int nm = p.nm, nw = p.nw, ncol = nm * nw;
  const int kk = p.panelKK[panel];
  const int b1p = p.panelB1[panel];

  // LDS carve-up
  T2v* X = reinterpret_cast<T2v*>(smem);                        // (groups, ncol)
  T2v* W = X + size_t(p.nG0) * ncol;                             // (m0, groups)
  const size_t xwBytes = (size_t(p.nG0) * ncol + size_t(p.m0) * p.nG0) * sizeof(T2v);
  double2* g3 = reinterpret_cast<double2*>(smem + (xwBytes + 15) / 16 * 16);  // 8 x ncol
  double2* sU2 = g3 + size_t(kSepRows) * ncol;                   // 8 x (nw * nb2max)
  double2* gp = sU2 + size_t(kSepRows) * nw * p.nb2max;          // 8 x (nm * nb2max)
  double* gs = reinterpret_cast<double*>(gp + size_t(kSepRows) * nm * p.nb2max);  // 8 x nm*nb2max
  double* se2 = gs + size_t(kSepRows) * nm * p.nb2max;           // 8 x nb2max
  double* sw3 = se2 + size_t(kSepRows) * p.nb2max;               // 8 x nm
  SepXShared* rinfo = reinterpret_cast<SepXShared*>(sw3 + size_t(kSepRows) * nm);  // m0
  int* list = reinterpret_cast<int*>(rinfo + p.m0);              // m0 + 1 (count at [m0])

  // ---- rows of the line and the screen
  for (int jx = t; jx < p.m0; jx += 256) {
    const int mesh = (jz * p.m1 + jy) * p.m0 + jx;
    int row = p.meshToRow[mesh];
    if (row < p.rowLo || row >= p.rowHi) row = -1;
    SepXShared ri{row, 0, 0, 0, 0};
    if (row >= 0) {
      ri.iq = mesh_diff_index(mesh, p.kkMesh[kk], p.m0, p.m1, p.m2);
      ri.nb2 = p.rowNb2[row];
      ri.u2off = p.rowU2off[row];
      ri.soff = p.rowStateOff[row];
      if (p.screen > 0.) {
        const double wlo = p.qWlo[ri.iq], whi = p.qWhi[ri.iq];
        const double e2lo = p.e2pool[ri.soff], e2hi = p.e2pool[ri.soff + ri.nb2 - 1];
        const double* e1 = p.e1pool + p.kkStateOff[kk] + p.panelGStart[panel];
        const double lim = screen_width(p, int(e1 - p.e1pool)) / p.invSigma;
        bool keep = false;
        if (whi >= wlo) {  // at least one mode above the cutoff
          for (int gi = 0; gi < p.panelGSize[panel]; ++gi) {
            const double a_lo = e1[gi] - e2hi + wlo, a_hi = e1[gi] - e2lo + whi;
            const double b_lo = e1[gi] - e2hi - whi, b_hi = e1[gi] - e2lo - wlo;
            keep |= (a_hi > -lim && a_lo < lim) || (b_hi > -lim && b_lo < lim);
          }
        }
        if (!keep) ri.row = -1;
      }
    }
    rinfo[jx] = ri;
  }
  const T2v* T2g = static_cast<const T2v*>(p.T2) + size_t(panel) * (p.t2PanelStride / 2);
  for (int i = t; i < p.nG0 * ncol; i += 256) {
    const int g = i / ncol, c = i % ncol;
    X[i] = T2g[((size_t(g) * p.m1 + jy) * p.m2 + jz) * ncol + c];
  }
  for (int i = t; i < p.m0 * p.nG0; i += 256) {
    const int jx = i / p.nG0, g = i % p.nG0;
    const double2 w = p.tw0[(jx * p.g0val[g]) % p.m0];
    W[i] = T2v{T(w.x), T(w.y)};
  }
  __syncthreads();
  if (t == 0) {
    int n = 0;
    for (int jx = 0; jx < p.m0; ++jx)
      if (rinfo[jx].row >= 0) list[n++] = jx;
    list[p.m0] = n;
  }
  __syncthreads();
  const int nkeep = list[p.m0];

  double part[kGMax][CM];
#pragma unroll
  for (int gi = 0; gi < kGMax; ++gi)
#pragma unroll
    for (int c = 0; c < CM; ++c) part[gi][c] = 0.;
  const int r = t >> 5, sub = t & 31;   // 32 threads per row in the epilogue
  const int nCalc = p.nCalc;
  const int gstart = p.panelGStart[panel], gsize = p.panelGSize[panel];
  const double* e1 = p.e1pool + p.kkStateOff[kk] + gstart;
  const double inv_g = 1. / double(float(gsize));

  for (int base = 0; base < nkeep; base += kSepRows) {
    // ---- g3 of the pass's rows (16 B of X per 8 complex FMAs)
    for (int c = t; c < ncol; c += 256) {
      double2 acc[kSepRows];
#pragma unroll
      for (int q = 0; q < kSepRows; ++q) acc[q] = make_double2(0., 0.);
      int jxs[kSepRows];
#pragma unroll
      for (int q = 0; q < kSepRows; ++q) jxs[q] = list[min(base + q, nkeep - 1)];
      for (int g = 0; g < p.nG0; ++g) {
        const T2v xv = X[g * ncol + c];
        const double xr = double(xv.x), xi = double(xv.y);
#pragma unroll
        for (int q = 0; q < kSepRows; ++q) {
          const T2v w = W[jxs[q] * p.nG0 + g];
          const double wr = double(w.x), wi = double(w.y);
          acc[q].x += wr * xr - wi * xi;
          acc[q].y += wr * xi + wi * xr;
        }
      }
#pragma unroll
      for (int q = 0; q < kSepRows; ++q) g3[q * ncol + c] = acc[q];
    }
    // ---- per-row prefetch: U2 and energies in LDS, e3 column / omega / Bose in registers
    const bool rowOn = base + r < nkeep;
    SepXShared ri{-1, 0, 0, 0, 0};
    if (rowOn) ri = rinfo[list[base + r]];
    const int nb2 = ri.row >= 0 ? ri.nb2 : 0;
    for (int i = sub; i < nw * nb2; i += 32) sU2[r * nw * p.nb2max + i] = p.U2pool[ri.u2off + i];
    if (sub < nb2) se2[r * p.nb2max + sub] = p.e2pool[ri.soff + sub];
    double2 e3c[NMX];
    double w3 = 0., n3[CM];
#pragma unroll
    for (int c = 0; c < CM; ++c) n3[c] = 0.;
    const bool modeOn = nb2 > 0 && sub < nm;
    if (modeOn) {
      const double2* e3 = p.E3pool + size_t(ri.iq) * nm * nm + size_t(nm) * sub;
#pragma unroll
      for (int nu = 0; nu < NMX; ++nu)
        if (nu < nm) e3c[nu] = e3[nu];
      w3 = p.Wpool[size_t(ri.iq) * nm + sub];
      sw3[r * nm + sub] = w3;
#pragma unroll
      for (int c = 0; c < CM; ++c)
        if (c < nCalc) n3[c] = p.bose[(size_t(ri.iq) * nm + sub) * nCalc + c];
    }
    __syncthreads();
    // ---- g'(nu, b2) = sum_w2 conj(U2(w2, b2)) g3(nu, w2), thread nu = sub
    if (modeOn) {
      const double2* gr = g3 + r * ncol + sub * nw;
      for (int b2 = 0; b2 < nb2; ++b2) {
        const double2* u = sU2 + r * nw * p.nb2max + nw * b2;
        double2 s = make_double2(0., 0.);
        for (int w2 = 0; w2 < nw; ++w2) {
          s.x += u[w2].x * gr[w2].x + u[w2].y * gr[w2].y;
          s.y += u[w2].x * gr[w2].y - u[w2].y * gr[w2].x;
        }
        gp[(r * nm + sub) * p.nb2max + b2] = s;
      }
    }
    __syncthreads();
    // ---- g(nu2, b2) = sum_nu e3(nu, nu2) g'(nu, b2), thread nu2 = sub; |g|^2 in registers
    double v[kSepNb2];
#pragma unroll
    for (int b = 0; b < kSepNb2; ++b) v[b] = 0.;
    if (modeOn) {
#pragma unroll
      for (int b2 = 0; b2 < kSepNb2; ++b2) {
        if (b2 < nb2) {
          double2 s = make_double2(0., 0.);
#pragma unroll
          for (int nu = 0; nu < NMX; ++nu)
            if (nu < nm) {
              const double2 x = gp[(r * nm + nu) * p.nb2max + b2];
              s.x += x.x * e3c[nu].x - x.y * e3c[nu].y;
              s.y += x.x * e3c[nu].y + x.y * e3c[nu].x;
            }
          v[b2] = s.x * s.x + s.y * s.y;
        }
      }
      if (!REDUCE) {
        const int nb1 = p.kkNb1[kk];
        for (int b2 = 0; b2 < nb2; ++b2)
          p.out[p.rowOutOff[ri.row] + b1p + size_t(nb1) * (b2 + size_t(nb2) * sub)] = v[b2];
      }
    }
    if (REDUCE) {
      // symmetrizeCoupling along b2 (scattering.cpp:1250-1284), in registers
      if (modeOn) {
        const double* e2r = se2 + r * p.nb2max;
        for (int b = 0; b < nb2;) {
          int deg = 0;
          for (int i = b; i < nb2; ++i) {
            if (fabs(e2r[b] - e2r[i]) < 1.0e-6) deg++;
            else break;
          }
          if (deg > 1) {
            double s = 0.;
#pragma unroll
            for (int i = 0; i < kSepNb2; ++i)
              if (i >= b && i < b + deg) s += v[i] / double(float(deg));
#pragma unroll
            for (int i = 0; i < kSepNb2; ++i)
              if (i >= b && i < b + deg) v[i] = s;
          }
          b += deg;
        }
      }
      // ... and along nu (scattering.cpp:1286-1316), through LDS when the modes are degenerate
      int mydeg = 1, mystart = sub;
      if (modeOn) {
        const double* wr = sw3 + r * nm;
        for (int s0 = 0; s0 < nm;) {
          int deg = 0;
          for (int i = s0; i < nm; ++i) {
            if (fabs(wr[s0] - wr[i]) < 1.0e-6) deg++;
            else break;
          }
          if (sub >= s0 && sub < s0 + deg) {
            mystart = s0;
            mydeg = deg;
          }
          s0 += deg;
        }
      }
      if (__syncthreads_or(mydeg > 1)) {
        if (modeOn)
          for (int b2 = 0; b2 < nb2; ++b2) gs[(r * nm + sub) * p.nb2max + b2] = v[b2];
        __syncthreads();
        if (modeOn && mydeg > 1)
          for (int b2 = 0; b2 < nb2; ++b2) {
            double s = 0.;
            for (int i = 0; i < mydeg; ++i) s += gs[(r * nm + mystart + i) * p.nb2max + b2] / double(float(mydeg));
#pragma unroll
            for (int b = 0; b < kSepNb2; ++b)
              if (b == b2) v[b] = s;
          }
      }
      // Gaussian-delta weights (el_scattering.cpp:277-380)
      if (modeOn && w3 >= p.cutoff) {
#pragma unroll
        for (int b2 = 0; b2 < kSepNb2; ++b2) {
          if (b2 >= nb2) break;
          const double en2 = se2[r * p.nb2max + b2];
          const double cpl = v[b2] * inv_g;
          const int is2 = ri.soff + b2;
#pragma unroll
          for (int gi = 0; gi < kGMax; ++gi) {
            if (gi >= gsize) break;
            double d1, d2;
            if (p.adaptive) {
              const AdaptiveWidth aw = adaptive_width(p, int(e1 - p.e1pool) + gi, is2);
              d1 = adaptive_delta(e1[gi] - en2 + w3, aw);
              d2 = adaptive_delta(e1[gi] - en2 - w3, aw);
            } else {
              d1 = gaussian_delta(e1[gi] - en2 + w3, p.invSigma, p.deltaPref);
              d2 = gaussian_delta(e1[gi] - en2 - w3, p.invSigma, p.deltaPref);
            }
            if (d1 <= 0. && d2 <= 0.) continue;
#pragma unroll
            for (int c = 0; c < CM; ++c) {
              if (c >= nCalc) break;
              const double f2 = p.fermi[size_t(c) * p.numStates + is2];
              part[gi][c] += cpl * ((f2 + n3[c]) * d1 + (1. - f2 + n3[c]) * d2) * p.norm / w3 *
                             3.14159265358979323846;
            }
          }
        }
      }
    }
    __syncthreads();
  }
  if (REDUCE) reduce_partials<CM>(p, L, smem, part);
}

inline size_t sep_x_lds_bytes(int elem, int nG0, int ncol, int m0, int nw, int nm, int nb2max) {
  const size_t t2 = 2 * size_t(elem);
  return (size_t(nG0) * ncol * t2 + size_t(m0) * nG0 * t2 + 15) / 16 * 16 +
         size_t(kSepRows) * (ncol + nw * nb2max + nm * nb2max) * sizeof(double2) +
         size_t(kSepRows) * (nm * nb2max + nb2max + nm) * sizeof(double) +
         size_t(m0) * sizeof(SepXShared) + size_t(m0 + 1) * sizeof(int) + 64;
}

// ---- last stage on MFMA
// Same result as k_sep_x.  Per workgroup (one (jy, jz) line of mesh points and
// one panel), the kept rows jx are compacted, then for every tile of 16 of them
//   g3(jx, c) = sum_g w_x^{jx n0(g)} T2(g, jy, jz, c)
// runs as two real GEMMs on v_mfma_*_16x16x4 in the transform precision,
// sharing B(2g + s, c) = (Re, Im) X(g, c):
//   Re g3 = A1 B with A1(m, 2g + s) = (Re w, -Im w),  Im g3 = A2 B with A2 = (Im w, Re w),
// w = w(jx_m, g) from a twiddle table in LDS, B straight from T2 (L2).  The epilogue gives
// TPR threads to each row (thread sub = mode nu).  Workgroups are ordered
// with the panels innermost, so that consecutive workgroups share the rows'
// U2 and the q-line's phonons in L2.
// kXmNt: complex column tiles (16 columns) per wave: 3 for nm * nw <= 192, 6 for <= 384
constexpr int kXmKsc = 3;   // MFMA k-steps per B chunk

struct SepXmRow {            // per kept row, staged in LDS
  int jx, row, iq, nb2, u2off, soff;
};

typedef short s16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// Orders LDS accesses between the lanes of one wavefront (no block barrier).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Row data of a 16-row tile into LDS: U2 (row r at sU2 + r * u2s, nw x nb2max),
// e2 (16 x nb2max), omega (16 x nm) and the electron occupations of the rows'
// states (nCalc x 16 x nb2max).  Every global load of a chunk is issued before
// the LDS stores, so a tile waits for one memory round trip, not one per
// element.  Needs 16 nb2max <= 256, 16 nm <= 512 and nCalc 16 nb2max <= 512.
__device__ inline void sep_xm_stage_rows(const CoupParams& p, const SepXmRow* rows, int m0r, int nr,
                                         int nw, int nm, int u2s, double2* sU2, double* se2,
                                         double* sw3, int* sg3, double* sf2) {
  const int t = threadIdx.x, nb2max = p.nb2max;
  const int ne = 16 * nb2max, nwv = 16 * nm, nf = p.nCalc * ne;
  double ev = 0., wv[2] = {0., 0.}, fv[2] = {0., 0.};
  int gv[2] = {0, 0};
  if (t < ne) {
    const int r = t / nb2max, b = t % nb2max;
    if (r < nr && b < rows[m0r + r].nb2) ev = p.e2pool[rows[m0r + r].soff + b];
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int i = t + 256 * u;
    if (i < nwv) {
      const int r = i / nm, nu = i % nm;
      if (r < nr) {
        wv[u] = p.Wpool[size_t(rows[m0r + r].iq) * nm + nu];
        gv[u] = p.qModeGrp[size_t(rows[m0r + r].iq) * nm + nu];
      }
    }
    if (i < nf) {
      const int c = i / ne, o = i % ne, r = o / nb2max, b = o % nb2max;
      if (r < nr && b < rows[m0r + r].nb2)
        fv[u] = p.fermi[size_t(c) * p.numStates + rows[m0r + r].soff + b];
    }
  }
  const int per = nw * nb2max, nU = 16 * per;
  for (int i0 = t; i0 < nU; i0 += 4 * 256) {
    double2 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = i0 + 256 * u;
      v[u] = make_double2(0., 0.);
      if (i < nU) {
        const int r = i / per, o = i % per;
        if (r < nr) {
          const SepXmRow& rr = rows[m0r + r];
          if (o < nw * rr.nb2) v[u] = p.U2pool[rr.u2off + o];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = i0 + 256 * u;
      if (i < nU) sU2[(i / per) * u2s + i % per] = v[u];
    }
  }
  if (t < ne) se2[t] = ev;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int i = t + 256 * u;
    if (i < nwv) {
      sw3[i] = wv[u];
      sg3[i] = gv[u];
    }
    if (i < nf) sf2[i] = fv[u];
  }
}

// Split-BF16 operands of v_mfma_f32_16x16x32_bf16: x ~ hi + lo with
// hi = bf16(x), lo = bf16(x - hi).
__device__ inline void bf16_split8(const float (&x)[8], bf16x8_t& hi, bf16x8_t& lo) {
  s16x8_t h8, l8;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const short h = bf16_bits(x[j]);
    h8[j] = h;
    l8[j] = bf16_bits(x[j] - bf16_value(h));
  }
  hi = __builtin_bit_cast(bf16x8_t, h8);
  lo = __builtin_bit_cast(bf16x8_t, l8);
}

// BF3: the x-stage GEMMs in split-BF16x3 (hi*hi + hi*lo + lo*hi on
// v_mfma_f32_16x16x32_bf16, FP32 accumulation); T must be float.
// BREG: the B operands of all k-steps (at most 12, i.e. 24 x-groups) are loaded
// once per work item, in the prologue, where their latency overlaps the row
// compaction; otherwise they are loaded per tile in chunks of KSB k-steps.
template <typename T, bool REDUCE, int NMX, int CM, bool BF3 = false, int kXmNt = 3, bool BREG = false>
__global__ void __launch_bounds__(256, 2) k_sep_xm(CoupParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef typename Vec2<T>::type T2v;
  typedef typename Mfma4<T>::acc_t acc_t;
  constexpr int TPR = NMX <= 16 ? 16 : 32;  // epilogue threads per row
  constexpr int RPP = 256 / TPR;            // rows per epilogue pass
  constexpr int KSB = (sizeof(T) == 4 && kXmNt <= 3) ? 12 : 3;  // k-steps of B held in registers
  const int nLinesYZ = p.m1 * p.m2;
  const int nTilesTot = p.nPanels * nLinesYZ;
  const int bid = blockIdx.x;
  const int perXcd = gridDim.x / 8;
  const int Lx = (bid % 8) * perXcd + bid / 8;
  if (Lx >= nTilesTot) return;
  const int yz = Lx / p.nPanels, panel = Lx % p.nPanels;
  const int slot = panel * nLinesYZ + yz;  // partial-sum slot (panel-major, as k_collect reads it)
  const int jy = yz % p.m1, jz = yz / p.m1;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, lr = lane & 15, lg = lane >> 4;
  if (p.gate && *p.gate == 0) return;
  if (p.slotOn && !p.slotOn[slot]) {
    if (REDUCE && p.slotZero && t < kGMax * kCMax) p.partial[size_t(slot) * kGMax * kCMax + t] = 0.;
    return;
  }
  // no row of the line passes the energy screen: zero partials, before any slab load
  if (p.keepMask && p.keepMask[slot] == 0ull) {
    if (REDUCE && t < kGMax * kCMax) p.partial[size_t(slot) * kGMax * kCMax + t] = 0.;
    return;
  }
  const int nm = p.nm, nw = p.nw, ncol = nm * nw;
  const int NWP = 2 * nw + 1, LDG = nm * NWP;  // g3 row layout: (nu, 2 w2 + ri), padded per nu
  const int kk = p.panelKK[panel];
  const int b1p = p.panelB1[panel];
  const int nG0 = p.nG0, nG0p = nG0 + 1;
  const int kkMesh = p.kkMesh[kk];

  // LDS carve-up
  SepXmRow* rows = reinterpret_cast<SepXmRow*>(smem);                          // m0
  int* wcnt = reinterpret_cast<int*>(rows + p.m0);                             // 8
  int* sg0 = wcnt + 8;                                                         // nG0
  T2v* stw = reinterpret_cast<T2v*>(smem + (size_t(p.m0) * sizeof(SepXmRow) + (8 + nG0) * sizeof(int) + 15) / 16 * 16);
  T2v* Wk = stw + p.m0;                                                        // m0 x nG0p
  unsigned char* dyn = reinterpret_cast<unsigned char*>(Wk + size_t(p.m0) * nG0p);
  dyn = smem + (size_t(dyn - smem) + 15) / 16 * 16;
  // Row strides of U2 and g' padded by one element: the 4 rows a wave serves
  // then start in different LDS banks.
  const int u2s = nw * p.nb2max + 1, gps = nm * p.nb2max + 1;
  T* g3 = reinterpret_cast<T*>(dyn);                                           // 16 x LDG
  double2* sU2 = reinterpret_cast<double2*>(dyn + (size_t(16) * LDG * sizeof(T) + 15) / 16 * 16);  // 16 x u2s
  double2* gp = sU2 + size_t(16) * u2s;                                        // RPP x gps
  double* se2 = reinterpret_cast<double*>(gp + size_t(RPP) * gps);             // 16 x nb2max
  double* sw3 = se2 + size_t(16) * p.nb2max;                                   // 16 x nm
  double* sf2 = sw3 + size_t(16) * nm;                                         // nCalc x 16 x nb2max
  double* se1 = sf2 + size_t(p.nCalc) * 16 * p.nb2max;                         // kGMax
  int* sg3 = reinterpret_cast<int*>(se1 + kGMax);                              // 16 x nm

  // twiddles and group coordinates
  for (int i = t; i < p.m0; i += 256) {
    const double2 d = p.tw0[i];
    stw[i] = T2v{T(d.x), T(d.y)};
  }
  for (int i = t; i < nG0; i += 256) sg0[i] = p.g0val[i];
  if (t < p.panelGSize[panel]) se1[t] = p.e1pool[p.kkStateOff[kk] + p.panelGStart[panel] + t];

  const T2v* X = static_cast<const T2v*>(p.T2) + size_t(panel) * (p.t2PanelStride / 2) +
                 (size_t(jy) * p.m2 + jz) * ncol;
  const size_t gStride = size_t(p.m1) * p.m2 * ncol;  // T2v elements between groups
  const int KS = (2 * nG0 + 3) / 4;                    // k-steps of 4 real K
  constexpr int KSR = BREG ? 12 : 1;
  T bAll[KSR][kXmNt];
  if constexpr (BREG) {
#pragma unroll
    for (int q = 0; q < KSR; ++q) {
      const int k = 4 * q + lg, g = k >> 1, kc = k & 1;
      const bool gOk = g < nG0;
#pragma unroll
      for (int j = 0; j < kXmNt; ++j) {
        const int c = (wave * kXmNt + j) * 16 + lr;
        T v = T(0);  // one component: 4-byte (FP32) loads, half the bytes of a complex load
        if (gOk && c < ncol) v = reinterpret_cast<const T*>(X)[2 * (size_t(g) * gStride + c) + kc];
        bAll[q][j] = v;
      }
    }
  }

  // ---- rows of the line, energy screen, compaction (ascending jx)
  int nkeep = 0;
  if (p.keepMask) {
    // kept rows from the screen kernel: one load per kept row
    const unsigned long long mask = p.keepMask[slot];
    nkeep = __popcll(mask);
    for (int jx = t; jx < p.m0; jx += 256)
      if ((mask >> jx) & 1ull) {
        const int mesh = (jz * p.m1 + jy) * p.m0 + jx;
        const int4 mr = p.meshRow[mesh];
        rows[__popcll(mask & ((1ull << jx) - 1ull))] =
            SepXmRow{jx, mr.x, mesh_diff_index(mesh, kkMesh, p.m0, p.m1, p.m2), mr.y, mr.z, mr.w};
      }
    __syncthreads();
  } else
  for (int j0 = 0; j0 < p.m0; j0 += 256) {
    const int jx = j0 + t;
    SepXmRow ri{jx, -1, 0, 0, 0, 0};    if (jx < p.m0) {
      const int mesh = (jz * p.m1 + jy) * p.m0 + jx;
      ri.iq = mesh_diff_index(mesh, kkMesh, p.m0, p.m1, p.m2);
      double wlo = 0., whi = 0.;
      if (p.screen > 0.) {
        wlo = p.qWlo[ri.iq];
        whi = p.qWhi[ri.iq];
      }
      int row = p.meshToRow[mesh];
      if (row < p.rowLo || row >= p.rowHi) row = -1;
      if (row >= 0) {
        ri.nb2 = p.rowNb2[row];
        ri.u2off = p.rowU2off[row];
        ri.soff = p.rowStateOff[row];
        bool keep = true;
        if (p.screen > 0.) {
          const double2 er = p.rowE2range[row];
          const double e2lo = er.x, e2hi = er.y;
          const double* e1 = p.e1pool + p.kkStateOff[kk] + p.panelGStart[panel];
          const double lim = screen_width(p, int(e1 - p.e1pool)) / p.invSigma;
          keep = false;
          if (whi >= wlo) {  // at least one mode above the cutoff
            for (int gi = 0; gi < p.panelGSize[panel]; ++gi) {
              const double a_lo = e1[gi] - e2hi + wlo, a_hi = e1[gi] - e2lo + whi;
              const double b_lo = e1[gi] - e2hi - whi, b_hi = e1[gi] - e2lo - wlo;
              keep |= (a_hi > -lim && a_lo < lim) || (b_hi > -lim && b_lo < lim);
            }
          }
        }
        if (keep) ri.row = row;
      }
    }
    const bool keep = ri.row >= 0;
    const unsigned long long mask = __ballot(keep);
    if (lane == 0) wcnt[wave] = __popcll(mask);
    __syncthreads();
    int off = nkeep, tot = 0;
    for (int w = 0; w < 4; ++w) {
      if (w < wave) off += wcnt[w];
      tot += wcnt[w];
    }
    if (keep) rows[off + __popcll(mask & ((1ull << lane) - 1ull))] = ri;
    nkeep += tot;
    __syncthreads();
  }
  if (t == 0 && p.keptRows && nkeep > 0) atomicAdd(p.keptRows, (unsigned long long)nkeep);
  if (nkeep == 0) {
    if (REDUCE) {
      double part[kGMax][CM];
      for (int gi = 0; gi < kGMax; ++gi)
        for (int c = 0; c < CM; ++c) part[gi][c] = 0.;
      reduce_partials<CM>(p, slot, smem, part);
    }
    return;
  }
  // twiddles of the kept rows: Wk(k, g) = w_x^{jx_k n0(g)}, zero column g = nG0 pads the K loop
  for (int i = t; i < nkeep * nG0p; i += 256) {
    const int k = i / nG0p, g = i % nG0p;
    Wk[i] = g < nG0 ? stw[(rows[k].jx * sg0[g]) % p.m0] : T2v{T(0), T(0)};
  }
  __syncthreads();

  double part[kGMax][CM];
#pragma unroll
  for (int gi = 0; gi < kGMax; ++gi)
#pragma unroll
    for (int c = 0; c < CM; ++c) part[gi][c] = 0.;
  const int nCalc = p.nCalc;
  const int gstart = p.panelGStart[panel], gsize = p.panelGSize[panel];
  const double* e1 = p.e1pool + p.kkStateOff[kk] + gstart;
  const double scrW = p.screen > 0. ? screen_width(p, int(e1 - p.e1pool)) : 0.;
  const double inv_g = 1. / double(float(gsize));

  for (int m0r = 0; m0r < nkeep; m0r += 16) {
    const int nr = min(16, nkeep - m0r);
    const bool rowOk = lr < nr;
    const T2v* wrow = Wk + size_t(m0r + (rowOk ? lr : 0)) * nG0p;
    // phonon eigenvector column, Bose factors of the epilogue row (r, mode sub)
    T2v e3c[NMX];
    double n3[CM];
    auto load_e3 = [&](int pr) {
      const int r = pr + t / TPR, sub = t % TPR;
#pragma unroll
      for (int c = 0; c < CM; ++c) n3[c] = 0.;
      if (r < nr && sub < nm) {
        const int iq = rows[m0r + r].iq;
        const T2v* e3 = static_cast<const T2v*>(p.E3T) + size_t(iq) * nm * nm + sub;
#pragma unroll
        for (int nu = 0; nu < NMX; ++nu)
          if (nu < nm) e3c[nu] = e3[nu * nm];
#pragma unroll
        for (int c = 0; c < CM; ++c)
          if (c < p.nCalc) n3[c] = p.bose[(size_t(iq) * nm + sub) * p.nCalc + c];
      }
    };
    // Cr = A1 B, Ci = A2 B with B(2g + s, c) = (Xr, Xi)(g, c), A1(m, 2g + s) = (Wr, -Wi),
    // A2(m, 2g + s) = (Wi, Wr); wave owns complex column tiles wave*kXmNt .. +kXmNt
    acc_t accr[kXmNt], acci[kXmNt];
#pragma unroll
    for (int j = 0; j < kXmNt; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) accr[j][i] = acci[j][i] = T(0);
    if constexpr (BF3) {
      sep_xm_stage_rows(p, rows, m0r, nr, nw, nm, u2s, sU2, se2, sw3, sg3, sf2);
      // gfx950's v_mfma_f32_16x16x32_bf16, 32 real K per step: lane (lr, lg)
      // holds groups g = 16 kb + 4 lg + h, h < 4, (Re, Im) each, in the A and
      // the B operand alike (the pairing of K slots is all the product needs)
      for (int kb = 0; kb < (2 * nG0 + 31) / 32; ++kb) {
        const int gA = 16 * kb + 4 * lg;
        float a1[8], a2[8];
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const T2v w = wrow[gA + h < nG0 ? gA + h : nG0];
          const bool on = rowOk && gA + h < nG0;
          a1[2 * h] = on ? w.x : 0.f;
          a1[2 * h + 1] = on ? -w.y : 0.f;
          a2[2 * h] = on ? w.y : 0.f;
          a2[2 * h + 1] = on ? w.x : 0.f;
        }
        bf16x8_t a1h, a1l, a2h, a2l;
        bf16_split8(a1, a1h, a1l);
        bf16_split8(a2, a2h, a2l);
#pragma unroll
        for (int j = 0; j < kXmNt; ++j) {
          const int c = (wave * kXmNt + j) * 16 + lr;
          float b[8];
#pragma unroll
          for (int h = 0; h < 4; ++h) {
            T2v x = T2v{0.f, 0.f};
            if (c < ncol && gA + h < nG0) x = X[size_t(gA + h) * gStride + c];
            b[2 * h] = x.x;
            b[2 * h + 1] = x.y;
          }
          bf16x8_t bh, bl;
          bf16_split8(b, bh, bl);
          accr[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1h, bh, accr[j], 0, 0, 0);
          accr[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1h, bl, accr[j], 0, 0, 0);
          accr[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1l, bh, accr[j], 0, 0, 0);
          acci[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2h, bh, acci[j], 0, 0, 0);
          acci[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2h, bl, acci[j], 0, 0, 0);
          acci[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2l, bh, acci[j], 0, 0, 0);
        }
      }
    } else if constexpr (BREG) {
      sep_xm_stage_rows(p, rows, m0r, nr, nw, nm, u2s, sU2, se2, sw3, sg3, sf2);
      // fully unrolled with a predicate (no early exit), so that bAll stays in registers
#pragma unroll
      for (int q = 0; q < KSR; ++q) {
        if (q < KS) {
          const int k = 4 * q + lg, g = k >> 1, kc = k & 1;
          const bool gOk = g < nG0;
          const T2v w = wrow[gOk ? g : nG0];
          const bool on = rowOk && gOk;
          const T a1 = on ? (kc ? -w.y : w.x) : T(0);
          const T a2 = on ? (kc ? w.x : w.y) : T(0);
#pragma unroll
          for (int j = 0; j < kXmNt; ++j) {
            accr[j] = Mfma4<T>::mac(a1, bAll[q][j], accr[j]);
            acci[j] = Mfma4<T>::mac(a2, bAll[q][j], acci[j]);
          }
        }
      }
    } else
    for (int kb = 0; kb < KS; kb += KSB) {
      // B operands of KSB k-steps straight from T2, then the MFMAs
      T bv[KSB][kXmNt];
#pragma unroll
      for (int q = 0; q < KSB; ++q) {
        const int k = 4 * (kb + q) + lg, g = k >> 1, kc = k & 1;
        const bool gOk = g < nG0 && kb + q < KS;
#pragma unroll
        for (int j = 0; j < kXmNt; ++j) {
          const int c = (wave * kXmNt + j) * 16 + lr;
          T v = T(0);  // one component of the complex element
          if (gOk && c < ncol) v = reinterpret_cast<const T*>(X)[2 * (size_t(g) * gStride + c) + kc];
          bv[q][j] = v;
        }
      }
      // the tile's row data into LDS while the B loads are in flight; the
      // previous tile's epilogue ended with a barrier
      if (kb == 0) sep_xm_stage_rows(p, rows, m0r, nr, nw, nm, u2s, sU2, se2, sw3, sg3, sf2);
#pragma unroll
      for (int q = 0; q < KSB; ++q) {
        if (kb + q < KS) {
          const int k = 4 * (kb + q) + lg, g = k >> 1, kc = k & 1;
          const bool gOk = g < nG0;
          const T2v w = wrow[gOk ? g : nG0];
          const bool on = rowOk && gOk;
          const T a1 = on ? (kc ? -w.y : w.x) : T(0);
          const T a2 = on ? (kc ? w.x : w.y) : T(0);
#pragma unroll
          for (int j = 0; j < kXmNt; ++j) {
            accr[j] = Mfma4<T>::mac(a1, bv[q][j], accr[j]);
            acci[j] = Mfma4<T>::mac(a2, bv[q][j], acci[j]);
          }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < kXmNt; ++j) {
      const int c = (wave * kXmNt + j) * 16 + lr;
      if (c < ncol) {
        const int nu = c / nw, w2 = c - nu * nw;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          T* dst = g3 + Mfma4<T>::row(lg, i) * LDG + nu * NWP + 2 * w2;
          dst[0] = accr[j][i];
          dst[1] = acci[j][i];
        }
      }
    }
    // the first pass's phonon data: loads in flight across the barrier and the
    // electron rotation, registers free during the staging and the MFMAs
    load_e3(0);
    __syncthreads();

    // ---- epilogue, RPP rows per pass (the first pass's phonon data was prefetched)
    for (int pr = 0; pr < 16; pr += RPP) {
      const int r = pr + t / TPR, sub = t % TPR, rl = t / TPR;
      const bool rowOn = r < nr;
      const SepXmRow ri = rows[m0r + (rowOn ? r : 0)];
      const int nb2 = rowOn ? ri.nb2 : 0;
      const bool modeOn = rowOn && sub < nm;
      if (pr > 0) load_e3(pr);
      const double w3 = modeOn ? sw3[r * nm + sub] : 0.;
      // g'(nu, b2) = sum_w2 conj(U2(w2, b2)) g3(nu, w2), thread nu = sub.  Each wave
      // owns whole rows from here on: only wave-level ordering is needed.
      if (modeOn) {
        const T* gr = g3 + r * LDG + sub * NWP;
        for (int b2 = 0; b2 < nb2; ++b2) {
          const double2* u = sU2 + size_t(r) * u2s + b2 * nw;
          double sx = 0., sy = 0.;
          for (int w2 = 0; w2 < nw; ++w2) {
            const double xr = double(gr[2 * w2]), xi = double(gr[2 * w2 + 1]);
            sx += u[w2].x * xr + u[w2].y * xi;
            sy += u[w2].x * xi - u[w2].y * xr;
          }
          gp[rl * gps + sub * p.nb2max + b2] = make_double2(sx, sy);
        }
      }
      wave_sync();
      // g(nu2, b2) = sum_nu e3(nu, nu2) g'(nu, b2), thread nu2 = sub; |g|^2 in registers
      double v[kSepNb2];
#pragma unroll
      for (int b = 0; b < kSepNb2; ++b) v[b] = 0.;
      if (modeOn) {
#pragma unroll
        for (int b2 = 0; b2 < kSepNb2; ++b2) {
          if (b2 < nb2) {
            double sx = 0., sy = 0.;
#pragma unroll
            for (int nu = 0; nu < NMX; ++nu)
              if (nu < nm) {
                const double2 x = gp[rl * gps + nu * p.nb2max + b2];
                const double er = double(e3c[nu].x), ei = double(e3c[nu].y);
                sx += x.x * er - x.y * ei;
                sy += x.x * ei + x.y * er;
              }
            v[b2] = sx * sx + sy * sy;
          }
        }
        if (!REDUCE) {
          const int nb1 = p.kkNb1[kk];
          for (int b2 = 0; b2 < nb2; ++b2)
            p.out[p.rowOutOff[ri.row] + b1p + size_t(nb1) * (b2 + size_t(nb2) * sub)] = v[b2];
        }
      }
      if (REDUCE) {
        // symmetrizeCoupling along b2 (scattering.cpp:1250-1284), in registers
        if (modeOn) {
          const double* e2r = se2 + r * p.nb2max;
          for (int b = 0; b < nb2;) {
            int deg = 0;
            for (int i = b; i < nb2; ++i) {
              if (fabs(e2r[b] - e2r[i]) < 1.0e-6) deg++;
              else break;
            }
            if (deg > 1) {
              double s2 = 0.;
#pragma unroll
              for (int i = 0; i < kSepNb2; ++i)
                if (i >= b && i < b + deg) s2 += v[i] / double(float(deg));
#pragma unroll
              for (int i = 0; i < kSepNb2; ++i)
                if (i >= b && i < b + deg) v[i] = s2;
            }
            b += deg;
          }
        }
        // ... and along nu (scattering.cpp:1286-1316), through LDS when modes are degenerate
        // the mode's degenerate group (consecutive modes within 1e-6 of the
        // group's first), tabulated per q at set-up
        int mydeg = 1, mystart = sub;
        if (modeOn) {
          const int grp = sg3[r * nm + sub];
          mystart = grp & 0xff;
          mydeg = grp >> 8;
        }
        if (__any(mydeg > 1)) {  // g' of the row is dead here: its slots hold |g|^2
          double* gs = reinterpret_cast<double*>(gp);
          wave_sync();
          if (modeOn)
            for (int b2 = 0; b2 < nb2; ++b2) gs[2 * (rl * gps + sub * p.nb2max + b2)] = v[b2];
          wave_sync();
          if (modeOn && mydeg > 1)
            for (int b2 = 0; b2 < nb2; ++b2) {
              double s2 = 0.;
              for (int i = 0; i < mydeg; ++i)
                s2 += gs[2 * (rl * gps + (mystart + i) * p.nb2max + b2)] / double(float(mydeg));
#pragma unroll
              for (int b = 0; b < kSepNb2; ++b)
                if (b == b2) v[b] = s2;
            }
        }
        // Gaussian-delta weights (el_scattering.cpp:277-380); b2 loop kept rolled
        if (modeOn && w3 >= p.cutoff) {
#pragma unroll 1
          for (int b2 = 0; b2 < nb2; ++b2) {
            double vb = 0.;
#pragma unroll
            for (int b = 0; b < kSepNb2; ++b)
              if (b == b2) vb = v[b];
            const double en2 = se2[r * p.nb2max + b2];
            const double cpl = vb * inv_g;
            const int is2 = ri.soff + b2;
#pragma unroll
            for (int gi = 0; gi < kGMax; ++gi) {
              if (gi >= gsize) break;
              double d1, d2;
              if (p.adaptive) {
                const AdaptiveWidth aw = adaptive_width(p, int(e1 - p.e1pool) + gi, is2);
                d1 = adaptive_delta(se1[gi] - en2 + w3, aw);
                d2 = adaptive_delta(se1[gi] - en2 - w3, aw);
              } else {
                const double x1 = se1[gi] - en2 + w3, x2 = se1[gi] - en2 - w3;
                // with the energy screen on, a pair whose both weights are below
                // exp(-screen^2) of the peak is skipped, as whole rows are
                if (p.screen > 0. && fmin(fabs(x1), fabs(x2)) * p.invSigma >= scrW)
                  continue;
                d1 = gaussian_delta(x1, p.invSigma, p.deltaPref);
                d2 = gaussian_delta(x2, p.invSigma, p.deltaPref);
              }
              if (d1 <= 0. && d2 <= 0.) continue;
#pragma unroll
              for (int c = 0; c < CM; ++c) {
                if (c >= nCalc) break;
                const double f2 = sf2[(c * 16 + r) * p.nb2max + b2];
                part[gi][c] += cpl * ((f2 + n3[c]) * d1 + (1. - f2 + n3[c]) * d2) * p.norm / w3 *
                               3.14159265358979323846;
              }
            }
          }
        }
      }
      wave_sync();  // the next pass reuses this wave's g' rows
    }
    __syncthreads();  // the next tile rewrites g3, U2, e2, omega
  }
  if (REDUCE) reduce_partials<CM>(p, slot, smem, part);
}


// ------------------------------------------------------------------ split last stage
// The last stage as two kernels with small footprints, for nw <= 16 and
// precomputed row masks: many more workgroups share a CU than with the fused
// k_sep_xm (about 65 KB of LDS and 255 VGPRs), which is bound by memory latency.
// g3 rows go through HBM, (slot, jx, col) with col = w2 nm + nu, and the
// epilogue (sep_epilogue.hpp) does the same operations on the same values, so
// the results equal the fused kernel's.

// x-stage: g3(row, (nu, w2)) = sum_g w_x^{jx n0(g)} T2(g; nu, w2) of every
// row kept by the slot's mask, stored at G3 (slot, jx) as complex T.
// ROT: the kernel also applies the electron rotation of the epilogue,
// g'(nu, b2) = sum_w2 conj(U2(w2, b2)) g3(nu, w2) in FP64 with w2 in order
// (the arithmetic of k_sep_ep2's phase A, on the same FP32 g3 values), and
// stores g' instead: complex FP64 at G3 (slot, jx, b2, nu), nb2max nm entries
// per row of which the row's nb2 nm are written.  At cfg2's 1.7 bands per
// inner point that is about a fifth of the bytes of g3.
template <typename T, int kXmNt, bool ROT = false>
__global__ void __launch_bounds__(256) k_sep_xg(CoupParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef typename Vec2<T>::type T2v;
  typedef typename Mfma4<T>::acc_t acc_t;
  const int nLinesYZ = p.m1 * p.m2;
  const int nTilesTot = p.nPanels * nLinesYZ;
  const int bid = blockIdx.x;
  const int perXcd = gridDim.x / 8;
  const int Lx = (bid % 8) * perXcd + bid / 8;
  if (Lx >= nTilesTot) return;
  const int yz = Lx / p.nPanels, panel = Lx % p.nPanels;
  const int slot = panel * nLinesYZ + yz;
  const int jy = yz % p.m1, jz = yz / p.m1;
  if (p.gate && *p.gate == 0) return;
  if (p.slotOn && !p.slotOn[slot]) return;
  const unsigned long long mask = p.keepMask[slot];
  if (mask == 0ull) return;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, lr = lane & 15, lg = lane >> 4;
  if (t == 0 && p.keptSlots) atomicAdd(p.keptSlots, 1ull);
  const int nm = p.nm, nw = p.nw, ncol = nm * nw;
  const int nG0 = p.nG0, nG0p = nG0 + 1;
  int* jxs = reinterpret_cast<int*>(smem);                                     // 64: kept rows, ascending
  int* snb = jxs + 64;                                                         // ROT: 64 band counts
  int* su2 = snb + 64;                                                         // ROT: 64 U2 offsets
  int* sg0 = su2 + 64;                                                         // nG0
  T2v* stw = reinterpret_cast<T2v*>(smem + (size_t(192 + nG0) * sizeof(int) + 15) / 16 * 16);  // m0
  T2v* Wk = stw + p.m0;                                                        // nkeep x nG0p
  T2v* sG = Wk + size_t(p.m0) * nG0p;  // ROT: one tile's g3, 16 rows x (nm (nw + 1) + 1)
  // ROT: the tile's U2, 16 rows x (nb2max x 16 + 1) complex FP64 (w2 fastest, zero beyond the
  // row's bands and nw), 16-byte aligned after sG
  const int us = p.nb2max * 16 + 1;
  double2* sUx = reinterpret_cast<double2*>(
      smem + (size_t(reinterpret_cast<unsigned char*>(sG + 16 * (nm * (nw + 1) + 1)) - smem) + 15) / 16 * 16);
  const T2v* X = static_cast<const T2v*>(p.T2) + size_t(panel) * (p.t2PanelStride / 2) +
                 (size_t(jy) * p.m2 + jz) * ncol;
  const size_t gStride = size_t(p.m1) * p.m2 * ncol;
  const int KS = (2 * nG0 + 3) / 4;  // <= 12, checked by the launcher
  T bAll[12][kXmNt];
#pragma unroll
  for (int q = 0; q < 12; ++q) {
    const int k = 4 * q + lg, g = k >> 1, kc = k & 1;
    const bool gOk = g < nG0;
#pragma unroll
    for (int j = 0; j < kXmNt; ++j) {
      const int c = (wave * kXmNt + j) * 16 + lr;
      T v = T(0);  // one component: 4-byte (FP32) loads, half the bytes of a complex load
      if (gOk && c < ncol) v = reinterpret_cast<const T*>(X)[2 * (size_t(g) * gStride + c) + kc];
      bAll[q][j] = v;
    }
  }
  for (int i = t; i < p.m0; i += 256) {
    const double2 d = p.tw0[i];
    stw[i] = T2v{T(d.x), T(d.y)};
  }
  for (int i = t; i < nG0; i += 256) sg0[i] = p.g0val[i];
  if (t < p.m0 && ((mask >> t) & 1ull)) {
    const int k = __popcll(mask & ((1ull << t) - 1ull));
    jxs[k] = t;
    if (ROT) {
      const int4 mr = p.meshRow[(jz * p.m1 + jy) * p.m0 + t];
      snb[k] = mr.y;
      su2[k] = mr.z;
    }
  }
  const int nkeep = __popcll(mask);
  __syncthreads();
  for (int i = t; i < nkeep * nG0p; i += 256) {
    const int k = i / nG0p, g = i % nG0p;
    Wk[i] = g < nG0 ? stw[(jxs[k] * sg0[g]) % p.m0] : T2v{T(0), T(0)};
  }
  __syncthreads();
  T2v* out = static_cast<T2v*>(p.G3) + size_t(slot) * p.m0 * ncol;
  // ROT: g' rows of nb2max nm complex FP64, (b2, nu) within a row
  const int gs = nw + 1, rs = nm * gs + 1, rowG = p.nb2max * nm;
  double2* outR = static_cast<double2*>(p.G3) + size_t(slot) * p.m0 * rowG;
  int sgOff[kXmNt];  // ROT: LDS offset of the lane's column (nu, w2) within a tile row
#pragma unroll
  for (int j = 0; j < kXmNt; ++j) {
    const int c = (wave * kXmNt + j) * 16 + lr;
    sgOff[j] = (c % nm) * gs + c / nm;  // T2's columns are (w2, nu)
  }
  for (int m0r = 0; m0r < nkeep; m0r += 16) {
    const int nr = min(16, nkeep - m0r);
    const bool rowOk = lr < nr;
    const T2v* wrow = Wk + size_t(m0r + (rowOk ? lr : 0)) * nG0p;
    acc_t accr[kXmNt], acci[kXmNt];
#pragma unroll
    for (int j = 0; j < kXmNt; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) accr[j][i] = acci[j][i] = T(0);
#pragma unroll
    for (int q = 0; q < 12; ++q) {
      if (q < KS) {
        const int k = 4 * q + lg, g = k >> 1, kc = k & 1;
        const bool gOk = g < nG0;
        const T2v w = wrow[gOk ? g : nG0];
        const bool on = rowOk && gOk;
        const T a1 = on ? (kc ? -w.y : w.x) : T(0);
        const T a2 = on ? (kc ? w.x : w.y) : T(0);
#pragma unroll
        for (int j = 0; j < kXmNt; ++j) {
          accr[j] = Mfma4<T>::mac(a1, bAll[q][j], accr[j]);
          acci[j] = Mfma4<T>::mac(a2, bAll[q][j], acci[j]);
        }
      }
    }
    if constexpr (ROT) {
      __syncthreads();  // the previous tile's rotation has read sG
#pragma unroll
      for (int j = 0; j < kXmNt; ++j) {
        const int c = (wave * kXmNt + j) * 16 + lr;
        if (c < ncol) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int row = Mfma4<T>::row(lg, i);
            if (row < nr) sG[row * rs + sgOff[j]] = T2v{accr[j][i], acci[j][i]};
          }
        }
      }
      // U2 of the tile's rows, each entry read from HBM once (not once per mode)
      for (int i = t; i < 16 * p.nb2max * 16; i += 256) {
        const int r = i / (p.nb2max * 16), o = i - r * (p.nb2max * 16), b2 = o >> 4, w2 = o & 15;
        double2 v = make_double2(0., 0.);
        if (r < nr && b2 < snb[m0r + r] && w2 < nw) v = p.U2pool[su2[m0r + r] + b2 * nw + w2];
        sUx[r * us + o] = v;
      }
      __syncthreads();
      // thread (row r, mode nu), nm <= 16 so 16 rows x nm <= 256 threads
      if (t < nr * nm) {
        const int r = t / nm, nu = t - r * nm, k = m0r + r;
        const int nb2 = snb[k];
        const double2* u = sUx + r * us;
        const T2v* x = sG + r * rs + nu * gs;
        double2* o = outR + size_t(jxs[k]) * rowG + nu;
        for (int b2 = 0; b2 < nb2; ++b2) {
          double ar = 0., ai = 0.;
#pragma unroll
          for (int w2 = 0; w2 < 16; ++w2) {
            if (w2 < nw) {
              const double2 c = u[b2 * 16 + w2];
              const double xr = double(x[w2].x), xi = double(x[w2].y);
              ar += c.x * xr + c.y * xi;
              ai += c.x * xi - c.y * xr;
            }
          }
          o[b2 * nm] = make_double2(ar, ai);
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < kXmNt; ++j) {
        const int c = (wave * kXmNt + j) * 16 + lr;
        if (c < ncol) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int row = Mfma4<T>::row(lg, i);
            if (row < nr) out[size_t(jxs[m0r + row]) * ncol + c] = T2v{accr[j][i], acci[j][i]};
          }
        }
      }
    }
  }
}

// rot: the x-stage with the electron rotation (a tile of g3 and its rows' U2 in LDS)
inline size_t sep_xg_lds_bytes(int elem, int nG0, int m0, int nm = 0, int nw = 0, bool rot = false,
                               int nb2max = 0) {
  size_t b = (size_t(192 + nG0) * sizeof(int) + 15) / 16 * 16 + size_t(m0) * (nG0 + 2) * 2 * elem;
  if (rot) b += (size_t(16) * (nm * (nw + 1) + 1) * 2 * elem + 15) / 16 * 16 +
                size_t(16) * (nb2max * 16 + 1) * sizeof(double2);
  return b + 64;
}

// The y-stage and the x-stage in one kernel, so that the x-stage slabs T2
// never go through HBM.  Workgroup (block of 16 columns, jz, panel): per tile
// of 16 y coordinates the y-stage (sep_y_tile) leaves T2 of every group in LDS,
// real and imaginary parts as rows k = 2g, 2g + 1, and the waves run the
// x-stage of the tile's slots in turn: g3(jx, c) = sum_k A(jx, k) B(k, c) on
// v_mfma_*_16x16x4 with A = the twiddles of the slot's kept rows, (Re w, Im w)
// at k = 2g and (-Im w, Re w) at 2g + 1, and write the kept rows' g3 for the
// block's columns.  The k order is that of k_sep_xg and k_sep_xm, so the g3
// are the same.
// Matrix cores and the g3 writes: cfg2's full launch (128 panels of 40^3 x 192
// columns) is 16 GFLOP FP64 in y (20 of 24 pair rows used), 80 GFLOP FP32 in x and
// 9 GB of traffic.  With the y sums as FMAs of four y coordinates per LDS read
// of T1, in threads that owned whole groups of uneven size, it took 3.9 ms; on
// the matrix cores 3.3 with a coordinate per row, 3.1 with conjugate pairs (FP64,
// 27 x 28 x 29: 1.94 and 1.88 ms).  Non-temporal g3 stores and the slots' masks in
// LDS measured the same.
template <typename T>
__global__ void __launch_bounds__(256) k_sep_yx(SepParams sp, CoupParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef typename Vec2<T>::type T2v;
  typedef typename Mfma4<T>::acc_t acc_t;
  const int cb = blockIdx.x, jz = blockIdx.y, panel = blockIdx.z;
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, lr = lane & 15,
            lg = lane >> 4;
  const int ncol = sp.ncol, my = sp.my, m0 = p.m0, nG0 = sp.nG0;
  const int KS = (2 * nG0 + 3) / 4, kp = 4 * KS;  // KS <= 12, checked by the launcher
  const int as = kp + 1, js = kp * 16 + 16;       // padded: rows in different banks
  const SepYShared sy = sep_y_stage(sp, smem, jz);
  T2v* sA = reinterpret_cast<T2v*>(smem + sep_y_lds_bytes(my, sp.nQuads));  // (jx, k): (a1, a2)
  T* sT2 = reinterpret_cast<T*>(sA + size_t(m0) * as);                      // (jj, k, 16 columns)
  int* sJx = reinterpret_cast<int*>(sT2 + size_t(16) * js) + wave * 64;     // kept rows of the wave's slot
  for (int i = t; i < m0 * kp; i += 256) {
    const int jx = i / kp, k = i - jx * kp, g = k >> 1;
    T2v a = T2v{T(0), T(0)};
    if (g < nG0) {
      const double2 d = p.tw0[(jx * p.g0val[g]) % m0];
      a = (k & 1) ? T2v{-T(d.y), T(d.x)} : T2v{T(d.x), T(d.y)};
    }
    sA[jx * as + k] = a;
  }
  for (int i = t; i < 16 * (kp - 2 * nG0) * 16; i += 256) {  // the padding of the last k-step
    const int r = i / 16, jj = r / (kp - 2 * nG0), k = 2 * nG0 + r % (kp - 2 * nG0);
    sT2[jj * js + k * 16 + (i & 15)] = T(0);
  }
  __syncthreads();
  const T2v* T1 = reinterpret_cast<const T2v*>(static_cast<const T*>(sp.T1) + size_t(panel) * sp.t1PanelStride);
  const int nLinesYZ = p.m1 * p.m2;
  const int c = cb * 16 + lr;
  for (int r0 = 0; r0 < sep_y_pairs(my); r0 += 8) {
    sep_y_tile<T>(sp, sy, T1, cb * 16, r0, [&](int g, int jj, double re, double im) {
      sT2[jj * js + (2 * g) * 16 + lr] = T(re);
      sT2[jj * js + (2 * g + 1) * 16 + lr] = T(im);
    });
    __syncthreads();
    const int np = min(8, sep_y_pairs(my) - r0);
    for (int i = wave; i < 2 * np; i += 4) {  // only the tile's pairs, so that the waves share them evenly
      const int jj = i < np ? i : 8 + i - np, jy = sep_y_coord(my, r0, jj);
      if (jy < 0) continue;
      const int slot = panel * nLinesYZ + jz * p.m1 + jy;
      const unsigned long long mask = p.keepMask[slot];
      if (mask == 0ull) continue;
      wave_sync();  // the wave's previous slot has read its list
      if (lane < m0 && ((mask >> lane) & 1ull)) sJx[__popcll(mask & ((1ull << lane) - 1ull))] = lane;
      wave_sync();
      const int nkeep = __popcll(mask);
      T b[12];
#pragma unroll
      for (int q = 0; q < 12; ++q)
        if (q < KS) b[q] = sT2[jj * js + (4 * q + lg) * 16 + lr];
      T2v* out = static_cast<T2v*>(p.G3) + size_t(slot) * m0 * ncol + c;
      for (int m0r = 0; m0r < nkeep; m0r += 16) {
        const int nr = min(16, nkeep - m0r);
        const T2v* arow = sA + sJx[min(m0r + lr, nkeep - 1)] * as + lg;
        acc_t accr, acci;
#pragma unroll
        for (int i = 0; i < 4; ++i) accr[i] = acci[i] = T(0);
#pragma unroll
        for (int q = 0; q < 12; ++q) {
          if (q < KS) {
            const T2v a = arow[4 * q];
            accr = Mfma4<T>::mac(a.x, b[q], accr);
            acci = Mfma4<T>::mac(a.y, b[q], acci);
          }
        }
        if (c < ncol) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int row = Mfma4<T>::row(lg, i);
            if (row < nr) out[size_t(sJx[m0r + row]) * ncol] = T2v{accr[i], acci[i]};
          }
        }
      }
    }
    __syncthreads();  // the next tile rewrites T2
  }
}

// ------------------------------------------------------------------ split epilogue
// Only what the epilogue of the split last stage reads.  A small block: the
// kernel keeps its scalars in SGPRs instead of spilling the full CoupParams'
// into VGPR lanes.
struct EpParams {
  const unsigned long long* keepMask;
  double* partial;  // (slot, kGMax, kCMax)
  const int* panelKK;
  const int* panelGStart;
  const int* panelGSize;
  const int* kkMesh;
  const int* kkStateOff;
  const int4* meshRow;     // per mesh point: (row, nb2, u2off, stateOff)
  const double* e1pool;
  const double* e2pool;
  const double* Wpool;     // (q, nu)
  const int* qModeGrp;     // (q, nu): first mode of the group | size << 8
  const double2* U2pool;
  const double* fermi;     // (calc, state)
  const double* bose;      // (q, nu, calc)
  const void* E3T;         // (q, nu, nu2) in the transform's precision
  const void* G3;          // (slot, jx, (w2, nu)) in the transform's precision; with the
                           // rotation done by the x-stage, (slot, jx, b2, nu) complex FP64
  const double* screenOf;  // per outer state: screen width of the panel its b1 group starts (null: screen)
  unsigned long long* keptRows;
  unsigned long long* keptBands;
  const unsigned char* slotOn;  // compute only slots with slotOn != 0 (null: all)
  const int* gate;              // run only when *gate != 0 (null: always)
  int slotZero;                 // slots off: 1 = write zero partials, 0 = leave them
  double invSigma, deltaPref, norm, cutoff, screen;
  int m0, m1, m2, nPanels, nm, nw, nCalc, numStates;
  int nb2max;              // g' rows of the rotating x-stage hold nb2max nm entries
  int rpw;                 // rows per pass: whole rows of nm lanes, rpw nm <= 64
  // adaptive smearing: group velocities of the states and the scaled cell (CoupParams)
  int adaptive;
  const double* stateV;
  double qT[9];
  double minWidth;
};

// The epilogue kernel (sep_epilogue.hpp) of `grid` slots on stream s: rows per
// pass and template instance by the mode count, band counts, b1 groups and
// calculations of the launch.  pre: G3 holds g' (FP32 data only).
template <typename T>
void launch_ep2(EpParams q, int gsizeMax, int grid, bool pre, hipStream_t s);

constexpr int kXminBlocks = 64;

// Closest approach to resonance of every panel of the chunk, for the energy
// screen widths: the minimum over the panel's rows (inner points of the
// range), their bands b2, the modes above the cutoff and the b1 group's
// energies e1 of |x| sigma, x = (e1 - e2 +- omega) / sigma, over the pairs
// with x <= 6 (the others have zero weight under the one-sided cut).  Grid (kXminBlocks, panels): block b
// takes mesh points b * 256 + t, strided by 256 * kXminBlocks.  A block first
// evaluates only the rows that pass the interval test at the configured
// width n: a row that fails it is at least n sigma from resonance in every
// pair, so once the block has found a pair closer than n the skipped rows
// cannot hold its minimum.  Otherwise it evaluates every row.  One partial
// minimum (energy units, HUGE_VAL when there is no pair) per block.
// Bound by the frequencies' loads: a wave lists its rows in LDS and then takes
// them (row, mode) by lane, so that a load's lanes read neighbouring modes.  With
// a row per lane each load touched 64 lines: 313 us against 199 for 128 panels of
// a 40^3 mesh of 12 modes, 12.7 against 10.3 for a line of a 9 x 8 x 7 mesh of 9.
static __global__ void __launch_bounds__(256) k_sep_xmin(CoupParams p) {
  const int panel = blockIdx.y, t = threadIdx.x, lane = t & 63;
  const int kk = p.panelKK[panel];
  const int kmesh = p.kkMesh[kk];
  const double* e1 = p.e1pool + p.kkStateOff[kk] + p.panelGStart[panel];
  const int gsz = p.panelGSize[panel];
  const double lim = p.screen / p.invSigma;
  const int nmesh = p.m0 * p.m1 * p.m2, nm = p.nm;
  __shared__ double red[256];
  __shared__ int4 list[256];  // per wave 64 rows: (q, first state, bands)
  int4* mine = list + (t & ~63);
  const float invNm = 1.f / float(nm);
  double best = HUGE_VAL, bmin = HUGE_VAL;
  for (int pass = 0; pass < 2; ++pass) {
    for (int m0 = blockIdx.x * 256 + (t & ~63); m0 < nmesh; m0 += 256 * kXminBlocks) {
      const int mesh = m0 + lane;
      int4 mr = make_int4(-1, 0, 0, 0);
      if (mesh < nmesh) mr = p.meshRow[mesh];
      bool keep = mr.x >= p.rowLo && mr.x < p.rowHi;
      int iq = 0;
      if (keep) {
        iq = mesh_diff_index(mesh, kmesh, p.m0, p.m1, p.m2);
        const double wlo = p.qWlo[iq], whi = p.qWhi[iq];
        keep = whi >= wlo;  // a mode above the cutoff
        if (keep && pass == 0) {
          const double2 er = p.rowE2range[mr.x];
          keep = false;
          for (int gi = 0; gi < gsz; ++gi) {
            const double a_lo = e1[gi] - er.y + wlo, a_hi = e1[gi] - er.x + whi;
            const double b_lo = e1[gi] - er.y - whi, b_hi = e1[gi] - er.x - wlo;
            keep |= (a_hi > -lim && a_lo < lim) || (b_hi > -lim && b_lo < lim);
          }
        }
      }
      const unsigned long long kept = __ballot(keep);
      wave_sync();  // the wave has read its previous list
      if (keep) mine[__popcll(kept & ((1ull << lane) - 1ull))] = make_int4(iq, mr.w, mr.y, 0);
      wave_sync();
      const int items = __popcll(kept) * nm;
      for (int i = lane; i < items; i += 64) {
        int r = int((float(i) + 0.5f) * invNm);  // i / nm, exact up to 64 rows
        const int4 row = mine[r];
        const double om = p.Wpool[size_t(row.x) * nm + (i - r * nm)];
        if (om < p.cutoff) continue;
        for (int b2 = 0; b2 < row.z; ++b2) {
          const double e2 = p.e2pool[row.y + b2];
          for (int gi = 0; gi < gsz; ++gi) {
            const double d = e1[gi] - e2;
            // only pairs the one-sided Gaussian can weigh (x <= 6, delta_function.cpp:43)
            const double a = d + om, b = d - om;
            if (a * p.invSigma <= 6.) best = fmin(best, fabs(a));
            if (b * p.invSigma <= 6.) best = fmin(best, fabs(b));
          }
        }
      }
    }
    red[t] = best;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
      if (t < s) red[t] = fmin(red[t], red[t + s]);
      __syncthreads();
    }
    bmin = red[0];
    __syncthreads();
    if (bmin < lim) break;  // block-uniform
  }
  if (t == 0) p.xminPart[size_t(panel) * kXminBlocks + blockIdx.x] = bmin;
}

// Screen width of a panel: sqrt(xmin^2 + n^2) sigma, with xmin its closest
// approach to resonance in units of sigma.  A pair that the screen drops then
// weighs at most exp(-n^2) of the panel's most resonant weighed pair, whatever
// the panel's distance to resonance (a panel whose pairs all lie in the
// Gaussian tails keeps its closest rows).  For a whole wave; the same value in
// every lane.
__device__ inline double sep_panel_width(const CoupParams& p, int panel) {
  double m = HUGE_VAL;
  for (int b = threadIdx.x & 63; b < kXminBlocks; b += 64) m = fmin(m, p.xminPart[size_t(panel) * kXminBlocks + b]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmin(m, __shfl_xor(m, o));
  const double x = m * p.invSigma;
  return x < HUGE_VAL ? sqrt(x * x + p.screen * p.screen) : p.screen;
}

// The widths alone (where no row masks are made).  One wave per panel.
static __global__ void __launch_bounds__(64) k_sep_xmin_fin(CoupParams p) {
  const int panel = blockIdx.x;
  const double w = sep_panel_width(p, panel);
  if (threadIdx.x == 0) p.screenOf[p.kkStateOff[p.panelKK[panel]] + p.panelGStart[panel]] = w;
}

// Row lists of the last stage: for every (panel, yz) slot, bit jx of
// keepMask[slot] is set when mesh point (jx, jy, jz) is an inner point of the
// range and passes the energy screen (same interval test as k_sep_x; every
// valid row when the screen is off), m0 <= 64.  A row per lane, 64, 32 or 16 lanes
// per slot; grid (slots of a panel, panels).  With widths per panel each wave
// works its panel's out, and the first stores it for the epilogue.  A slot per
// thread reads its rows one after the other from lines of its own: 144 us for 128
// panels of a 40^3 mesh against 101, and 14 against 5 for 128 panels of a 12^3 one.
template <int L>
__global__ void __launch_bounds__(256) k_sep_screen(CoupParams p) {
  const int nLinesYZ = p.m1 * p.m2, panel = blockIdx.y, t = threadIdx.x, jx = t % L;
  const int yz = blockIdx.x * (256 / L) + t / L;
  const int kk = p.panelKK[panel];
  const int gstart = p.panelGStart[panel], gsz = p.panelGSize[panel];
  const double* e1 = p.e1pool + p.kkStateOff[kk] + gstart;
  double lim = 0.;
  if (p.screen > 0.) {
    lim = p.screenOf ? sep_panel_width(p, panel) : p.screen;
    if (p.screenOf && t == 0 && blockIdx.x == 0) p.screenOf[p.kkStateOff[kk] + gstart] = lim;
    lim /= p.invSigma;
  }
  bool keep = false;
  if (yz < nLinesYZ && jx < p.m0) {
    const int mesh = yz * p.m0 + jx, row = p.meshRow[mesh].x;
    keep = row >= p.rowLo && row < p.rowHi;
    if (keep && p.screen > 0.) {
      const int iq = mesh_diff_index(mesh, p.kkMesh[kk], p.m0, p.m1, p.m2);
      const double wlo = p.qWlo[iq], whi = p.qWhi[iq];
      const double2 er = p.rowE2range[row];
      keep = false;
      if (whi >= wlo)  // at least one mode above the cutoff
        for (int gi = 0; gi < gsz; ++gi) {
          const double a_lo = e1[gi] - er.y + wlo, a_hi = e1[gi] - er.x + whi;
          const double b_lo = e1[gi] - er.y - whi, b_hi = e1[gi] - er.x - wlo;
          keep |= (a_hi > -lim && a_lo < lim) || (b_hi > -lim && b_lo < lim);
        }
    }
  }
  const unsigned long long all = __ballot(keep), ones = L == 64 ? ~0ull : (1ull << (L & 63)) - 1ull;
  if (jx == 0 && yz < nLinesYZ) p.keepMask[size_t(panel) * nLinesYZ + yz] = (all >> ((t & 63) / L * L)) & ones;
}

inline size_t sep_xm_lds_bytes(int elem, int nG0, int m0, int nw, int nm, int nb2max, int rpp, int nCalc) {
  auto up = [](size_t b) { return (b + 15) / 16 * 16; };
  size_t b = up(size_t(m0) * sizeof(SepXmRow) + (8 + nG0) * sizeof(int));
  b = up(b + size_t(m0) * 2 * elem + size_t(m0) * (nG0 + 1) * 2 * elem);
  const size_t g3 = std::max(size_t(16) * nm * (2 * nw + 1) * elem, size_t(rpp) * nm * nb2max * sizeof(double));
  b += up(g3);
  b += size_t(16) * (nw * nb2max + 1) * sizeof(double2) + size_t(rpp) * (nm * nb2max + 1) * sizeof(double2) +
       size_t(16) * nb2max * sizeof(double) + size_t(16) * nm * sizeof(double) +
       size_t(nCalc) * 16 * nb2max * sizeof(double) + size_t(kGMax) * sizeof(double) +
       size_t(16) * nm * sizeof(int);
  return std::max(b, size_t(kGMax) * kCMax * 4 * sizeof(double)) + 64;
}

// maxLineE: largest number of entries of a line (LDS sizing).
template <typename T>
void launch_separable_zy(const SepParams& sp, int maxLineE, hipStream_t s, bool yStage = true) {
  if (sp.nPanels <= 0) return;
  const size_t ldsZ = sep_stage_lds_bytes(sizeof(T), maxLineE, sp.ncol, sp.mz);
  const size_t ldsY = sep_y_lds_bytes(sp.my, sp.nQuads);
  PHX_REQUIRE(ldsZ <= 160 * 1024 && ldsY <= 160 * 1024, "separable transform: LDS budget exceeded");
  PHX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_sep_z<T>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, int(std::max<size_t>(ldsZ, 16))));
  PHX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_sep_y<T>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, int(std::max<size_t>(ldsY, 16))));
  hipLaunchKernelGGL(k_sep_z<T>, dim3(sp.nLines, sp.nPanels), dim3(256), ldsZ, s, sp);
  PHX_HIP(hipGetLastError());
  if (!yStage) return;  // the x-stage kernel runs the y-stage itself (k_sep_yx)
  hipLaunchKernelGGL(k_sep_y<T>, dim3(ceil_div(sp.ncol, 16), sp.mz, sp.nPanels), dim3(256), ldsY, s, sp);
  PHX_HIP(hipGetLastError());
}

// Where the split last stage's epilogue kernel runs: on the launch's stream
// (ep null), or on the stream ep once the x-stage kernel is done, so that it
// overlaps the work enqueued on the launch's stream after it.
struct EpFork {
  hipStream_t ep = nullptr;
  hipEvent_t xgDone = nullptr;   // recorded on the launch's stream after the x-stage kernel (ep set)
  hipEvent_t epStart = nullptr;  // timing: recorded on the epilogue's stream before it (null: off)
  hipEvent_t xgStart = nullptr;  // timing: recorded on the launch's stream right before the x-stage kernel
};

// mid (optional): recorded between the x-stage and the epilogue kernel when
// the last stage runs split.  Returns whether it did (then the epilogue ran
// on fork.ep when that is set).
template <typename T>
bool launch_separable_x(const SepParams& sp, const CoupParams& p, bool reduce, hipStream_t s,
                        hipEvent_t mid, const EpFork& fork = EpFork{}) {
  PHX_REQUIRE(p.nm <= kSepNm && p.nb2max <= kSepNb2,
              "separable transform supports nm <= 32 and at most 8 bands per inner point");
  // what the host chose (last_stage), whose stages before this one and buffers depend on it
  const bool split = p.stage != kStageFused;
  PHX_REQUIRE(split == (sp.modeFast != 0), "separable transform: column order of the split last stage");
  PHX_REQUIRE(!split || (reduce && p.G3 && p.keepMask && p.nw <= 16 && p.nG0 <= kSplitGroups && sp.ncol <= kSplitCols),
              "separable transform: the split last stage does not take these sizes");
  PHX_REQUIRE(p.stage == kStageYx || p.T2, "separable transform: x-stage without the y-stage's output");
  if (sp.nPanels <= 0) return false;
  const int tiles = sp.nPanels * sp.my * sp.mz;
  const int grid = ceil_div(tiles, 8) * 8;
  const int nmb = p.nm <= 12 ? 12 : p.nm <= 16 ? 16 : p.nm <= 24 ? 24 : kSepNm;
  const bool one = p.nCalc == 1;
  constexpr bool bf3t = sizeof(T) == 4;  // split-BF16x3 exists for the FP32 data path
  const bool bf3 = p.bf16x3 != 0;
  constexpr bool bregt = sizeof(T) == 4;  // B in registers for the whole item: FP32, <= 24 x-groups
  const bool breg = bregt && (2 * p.nG0 + 3) / 4 <= 12;
  PHX_REQUIRE(!bf3 || (bf3t && reduce && sp.ncol <= kSplitCols),
              "split-BF16x3: FP32 data, the linewidth reduction and nm nw <= 384");
  if (reduce && p.screen > 0. && p.screenOf) {
    PHX_REQUIRE(p.xminPart && p.meshRow, "energy screen: closest-approach buffers missing");
    hipLaunchKernelGGL(k_sep_xmin, dim3(kXminBlocks, sp.nPanels), dim3(256), 0, s, p);
    PHX_HIP(hipGetLastError());
    if (!(p.keepMask && sp.ncol <= kSplitCols)) {  // else the row masks' kernel stores the widths
      hipLaunchKernelGGL(k_sep_xmin_fin, dim3(sp.nPanels), dim3(64), 0, s, p);
      PHX_HIP(hipGetLastError());
    }
  }
  if (reduce && sp.ncol <= kSplitCols) {
    const bool wide = sp.ncol > kXgCols;
    const size_t ldsXm = sep_xm_lds_bytes(sizeof(T), p.nG0, p.m0, p.nw, p.nm, p.nb2max, nmb <= 16 ? 16 : 8,
                                             p.nCalc);
    PHX_REQUIRE(ldsXm <= 160 * 1024, "separable transform: LDS budget exceeded");
    PHX_REQUIRE(p.qModeGrp && p.E3T, "separable transform: mode-group or eigenvector table missing");
    if (p.keepMask) {
      PHX_REQUIRE(p.m0 <= 64 && p.meshRow, "separable transform: row masks need m0 <= 64");
      const int lines = sp.my * sp.mz;
      if (p.m0 <= 16) hipLaunchKernelGGL(k_sep_screen<16>, dim3(ceil_div(lines, 16), sp.nPanels), dim3(256), 0, s, p);
      else if (p.m0 <= 32)
        hipLaunchKernelGGL(k_sep_screen<32>, dim3(ceil_div(lines, 8), sp.nPanels), dim3(256), 0, s, p);
      else hipLaunchKernelGGL(k_sep_screen<64>, dim3(ceil_div(lines, 4), sp.nPanels), dim3(256), 0, s, p);
      PHX_HIP(hipGetLastError());
    }
    if (split) {
      if (fork.xgStart) PHX_HIP(hipEventRecord(fork.xgStart, s));
      const bool rot = p.stage == kStageRot;
      PHX_REQUIRE(p.stage == kStageYx || (sizeof(T) == 4 && sp.ncol <= kXgCols && p.nm <= 16 && !(rot && p.adaptive)),
                  "separable transform: the x-stage kernel does not take these sizes");
      if (p.stage == kStageYx) {
        PHX_REQUIRE(!p.slotOn && !p.gate, "separable transform: fused y/x-stage without slot masks");
        const size_t ldsYX = sep_yx_lds_bytes(sizeof(T), sp.nQuads, sp.my, sp.nG0, p.m0);
        PHX_REQUIRE(ldsYX <= 160 * 1024, "separable transform: LDS budget exceeded");
        PHX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_sep_yx<T>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, int(ldsYX)));
        hipLaunchKernelGGL(k_sep_yx<T>, dim3(ceil_div(sp.ncol, 16), sp.mz, sp.nPanels), dim3(256), ldsYX, s, sp, p);
      } else if constexpr (sizeof(T) == 4) {
        const size_t ldsA = sep_xg_lds_bytes(sizeof(T), p.nG0, p.m0, p.nm, p.nw, rot, p.nb2max);
        PHX_REQUIRE(ldsA <= 160 * 1024, "separable transform: LDS budget exceeded");
        auto xg = [&](auto kern) {
          PHX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, int(ldsA)));
          hipLaunchKernelGGL(kern, dim3(grid), dim3(256), ldsA, s, p);
        };
        if (rot) xg(k_sep_xg<T, 3, true>);
        else xg(k_sep_xg<T, 3, false>);
      }
      PHX_HIP(hipGetLastError());
      if (mid) PHX_HIP(hipEventRecord(mid, s));
      hipStream_t se = s;
      if (fork.ep) {
        PHX_HIP(hipEventRecord(fork.xgDone, s));
        PHX_HIP(hipStreamWaitEvent(fork.ep, fork.xgDone, 0));
        se = fork.ep;
      }
      if (fork.epStart) PHX_HIP(hipEventRecord(fork.epStart, se));
      EpParams q{};
      q.keepMask = p.keepMask;
      q.partial = p.partial;
      q.panelKK = p.panelKK;
      q.panelGStart = p.panelGStart;
      q.panelGSize = p.panelGSize;
      q.kkMesh = p.kkMesh;
      q.kkStateOff = p.kkStateOff;
      q.meshRow = p.meshRow;
      q.e1pool = p.e1pool;
      q.e2pool = p.e2pool;
      q.Wpool = p.Wpool;
      q.qModeGrp = p.qModeGrp;
      q.U2pool = p.U2pool;
      q.fermi = p.fermi;
      q.bose = p.bose;
      q.E3T = p.E3T;
      q.G3 = p.G3;
      q.screenOf = p.screenOf;
      q.keptRows = p.keptRows;
      q.keptBands = p.keptBands;
      q.slotOn = p.slotOn;
      q.gate = p.gate;
      q.slotZero = p.slotZero;
      q.invSigma = p.invSigma;
      q.deltaPref = p.deltaPref;
      q.norm = p.norm;
      q.cutoff = p.cutoff;
      q.screen = p.screen;
      q.m0 = p.m0;
      q.m1 = p.m1;
      q.m2 = p.m2;
      q.nPanels = p.nPanels;
      q.nm = p.nm;
      q.nw = p.nw;
      q.nCalc = p.nCalc;
      q.numStates = p.numStates;
      q.nb2max = p.nb2max;
      q.adaptive = p.adaptive;
      q.stateV = p.stateV;
      for (int i = 0; i < 9; ++i) q.qT[i] = p.qT[i];
      q.minWidth = p.minWidth;
      launch_ep2<T>(q, p.gsizeMax, grid, rot, se);
      return true;
    }
    auto go = [&](auto kern) {
      PHX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, int(ldsXm)));
      hipLaunchKernelGGL(kern, dim3(grid), dim3(256), ldsXm, s, p);
    };
#define PHX_XM(NMX)                                                                 \
    if (nmb == NMX) {                                                               \
      if (wide) {                                                                   \
        if (bf3 && one) go(k_sep_xm<T, true, NMX, 1, bf3t, 6>);                      \
        else if (bf3) go(k_sep_xm<T, true, NMX, kCMax, bf3t, 6>);                    \
        else if (one) go(k_sep_xm<T, true, NMX, 1, false, 6>);                       \
        else go(k_sep_xm<T, true, NMX, kCMax, false, 6>);                            \
      } else {                                                                      \
        if (bf3 && one) go(k_sep_xm<T, true, NMX, 1, bf3t>);                         \
        else if (bf3) go(k_sep_xm<T, true, NMX, kCMax, bf3t>);                       \
        else if (breg && one) go(k_sep_xm<T, true, NMX, 1, false, 3, bregt>);        \
        else if (breg) go(k_sep_xm<T, true, NMX, kCMax, false, 3, bregt>);           \
        else if (one) go(k_sep_xm<T, true, NMX, 1>);                                 \
        else go(k_sep_xm<T, true, NMX, kCMax>);                                      \
      }                                                                             \
    }
    PHX_XM(12) PHX_XM(16) PHX_XM(24) PHX_XM(32)
#undef PHX_XM
    PHX_HIP(hipGetLastError());
    return false;
  }
  PHX_REQUIRE(!p.slotOn && !p.gate, "separable transform: slot masks need nm nw <= 384");
  const size_t ldsX = std::max(sep_x_lds_bytes(sizeof(T), p.nG0, sp.ncol, p.m0, p.nw, p.nm, p.nb2max),
                               size_t(kGMax) * kCMax * 4 * sizeof(double));
  PHX_REQUIRE(ldsX <= 160 * 1024, "separable transform: LDS budget exceeded");
  auto go = [&](auto kern) {
    PHX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                hipFuncAttributeMaxDynamicSharedMemorySize, int(ldsX)));
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), ldsX, s, p);
  };
  const int nmo = p.nm <= 12 ? 12 : p.nm <= 18 ? 18 : kSepNm;
  if (reduce) {
    if (nmo == 12) one ? go(k_sep_x<T, true, 12, 1>) : go(k_sep_x<T, true, 12, kCMax>);
    else if (nmo == 18) one ? go(k_sep_x<T, true, 18, 1>) : go(k_sep_x<T, true, 18, kCMax>);
    else one ? go(k_sep_x<T, true, kSepNm, 1>) : go(k_sep_x<T, true, kSepNm, kCMax>);
  } else {
    if (nmo == 12) go(k_sep_x<T, false, 12, 1>);
    else if (nmo == 18) go(k_sep_x<T, false, 18, 1>);
    else go(k_sep_x<T, false, kSepNm, 1>);
  }
  PHX_HIP(hipGetLastError());
  return false;
}

}  // namespace phx
