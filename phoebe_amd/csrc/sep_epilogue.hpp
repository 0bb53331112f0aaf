// Epilogue of the split separable last stage (the EpParams of coupling_kernel.hpp),
// instantiated per precision in coupling_ep_f64.hip and coupling_ep_f32.hip.
#pragma once

#include "coupling_kernel.hpp"

namespace phx {

// Kept row of a slot, staged in LDS.
struct EpRow {
  int jxnb, iq, u2off, soff;  // jx | nb2 << 8
};

// Epilogue of the rows k_sep_yx / k_sep_xg wrote, one wave per slot (panel, yz
// line), passes of rpw rows with lane (row r, mode sub):
//   A  electron rotation g'(nu, b2) = sum_w2 conj(U2(w2, b2)) g3(nu, w2),
//      nu = sub, each g3 value converted once (outer loop over w2, NB
//      accumulators), U2 of the pass in LDS;
//   B  phonon rotation g(nu2, b2) = sum_nu e3(nu, nu2) g'(nu, b2), nu2 = sub,
//      the eigenvector column in registers, then |g|^2 and symmetrizeCoupling
//      along b2 (scattering.cpp:1250-1284) on the lane's own entries;
//   C  symmetrizeCoupling along nu (:1286-1316) from the group's entries and
//      the smearing weights of el_scattering.cpp:277-380 into per-lane
//      partial sums (CM calculations, GM members of the b1 group).
// Phases A and B run the pass's largest band count for every row (uniform
// branches; what a row computes beyond its own count is never read).  NB2 >=
// nb2max is the LDS stride of a row's bands, NMX >= nm the eigenvector column
// length.
// Bound by latency (the passes of a slot follow each other in one wave) and by
// LDS reads.  Each operand of the next pass is loaded into the registers of
// the present one as soon as a phase has used them up (g3 and U2 after A, e3
// after B), so part of its latency passes behind the other phases; the loads
// are unconditional (rows beyond the slot's read its last one), because a load
// under a branch makes the compiler wait for every load in flight.  cfg2's full
// launch (128 panels, 4 million rows of 12 modes, 16 bands x 1.7): 2.37 ms; 2.43
// with the rows in mesh order and column length rounded up to 16 modes (an exact
// one drops a quarter of phase B there), 2.5 with w2 fastest in g3 and all loads
// at a pass's start.  With k_sep_yx
// against the fused k_sep_xm and its y-stage, ms per pass: FP64, 12 modes x 16
// bands, 6 lines of a 27 x 28 x 29 mesh 6.3 against 21.2; FP32, 18 x 16, 4 lines
// of a 32^3 mesh 7.2 against 21.8.

// Phase A for NB bands: g'(nu, b2) = sum_w2 conj(U2(w2, b2)) g3(nu, w2) for the
// lane's mode, w2 in order.  No branches inside: entries beyond nw are zero in
// U2 and finite in g (a copy of the last one).
template <typename T2v, int NWX, int NB>
__device__ __forceinline__ void ep2_rot_el(const T2v (&g)[NWX], const double2* u, double2* out) {
  double ar[NB], ai[NB];
#pragma unroll
  for (int b2 = 0; b2 < NB; ++b2) ar[b2] = ai[b2] = 0.;
#pragma unroll
  for (int w2 = 0; w2 < NWX; ++w2) {
    auto gx = g[w2].x, gy = g[w2].y;
    asm volatile("" : "+v"(gx), "+v"(gy));  // converted here, not all ahead of the band loop
    const double xr = double(gx), xi = double(gy);
#pragma unroll
    for (int b2 = 0; b2 < NB; ++b2) {
      const double2 c = u[b2 * NWX + w2];
      ar[b2] += c.x * xr + c.y * xi;
      ai[b2] += c.x * xi - c.y * xr;
    }
  }
#pragma unroll
  for (int b2 = 0; b2 < NB; ++b2) out[b2] = make_double2(ar[b2], ai[b2]);
}

// Phase B for NB bands: g(nu2, b2) = sum_nu e3(nu, nu2) g'(nu, b2) for the
// lane's mode nu2, nu in order, and |g|^2.  Modes beyond nm count as zero (e3
// here, g' in its padding).
template <typename T2v, int NMX, int NB2, int NB>
__device__ __forceinline__ void ep2_rot_ph(const T2v (&e3c)[NMX], const double2* x, double* own) {
  double gr[NB], gi[NB];
#pragma unroll
  for (int b2 = 0; b2 < NB; ++b2) gr[b2] = gi[b2] = 0.;
#pragma unroll
  for (int nu = 0; nu < NMX; ++nu) {
    auto ex = e3c[nu].x, ey = e3c[nu].y;
    asm volatile("" : "+v"(ex), "+v"(ey));  // converted here, not all ahead of the band loop
    const double er = double(ex), ei = double(ey);
    const double2* xn = x + nu * NB2;
#pragma unroll
    for (int b2 = 0; b2 < NB; ++b2) {
      const double2 v = xn[b2];
      gr[b2] += v.x * er - v.y * ei;
      gi[b2] += v.x * ei + v.y * er;
    }
  }
#pragma unroll
  for (int b2 = 0; b2 < NB; ++b2) own[b2] = gr[b2] * gr[b2] + gi[b2] * gi[b2];
}

// Instances that serve one mode count only (1 to 6 atoms): the modes' offsets are
// then constants of the load instructions.
constexpr bool ep2_exact(int nmx) { return nmx <= 18; }

// FP32 rows of more than 4 bands whose U2 goes through registers: twice the U2
// entries and |g|^2, so 256 registers at two waves per SIMD (at 168 they spill 36
// to 183, which also cost more than the third wave gives).
constexpr bool ep2_wide(int elem, int nb2, bool pre) { return elem == 4 && nb2 > 4 && !pre; }
constexpr int ep2_waves(int elem, int nb2, bool pre) { return elem == 4 && !ep2_wide(elem, nb2, pre) ? 3 : 2; }

// Rows per pass at most: whole rows of nm lanes for the least nm served with
// NMX, and no more than five, or with up to 9 modes in the wide form 8, 6 or 7,
// as many as pay.  Ten rows of 6 modes fill the wave but hold twice the U2 entries
// in registers, and spill: 52 us against 37 per launch of 128 panels on a 12^3
// mesh.  Wide form, 8 bands, 200 points against a 16 x 17 x 16 mesh, adaptive, one and
// four calculations (three waves and five rows; two waves; the epilogue of one
// thread per row and mode that adaptive widths had before), ms: 3 modes 12.0 and
// 15.5; 9.3 and 9.7; 9.7 and 11.1.  6 modes 14.7 and 18.7; 11.6 and 12.1; 11.5 and
// 12.9.  9 modes (14^3) 11.1 and 15.0; 9.5 and 10.0; 9.5 and 12.3.  12 modes 21.6
// and 28.2; 19.2 and 19.8; 20.7 and 24.7.
constexpr int ep2_rows_max(int nmx, bool wide) {
  if (wide && nmx <= 9) return nmx <= 3 ? 8 : nmx <= 6 ? 6 : 7;
  return nmx <= 12 ? 5 : nmx <= 18 ? 4 : nmx <= 24 ? 3 : 2;
}

template <typename T, int CM, int NMX, int GM, int NB2, bool PRE, bool ADAPT>
__global__ void __launch_bounds__(64, ep2_waves(sizeof(T), NB2, PRE)) k_sep_ep2(EpParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef typename Vec2<T>::type T2v;
  constexpr int NWX = 16;
  constexpr int U2S = NWX * NB2 + 1;  // double2 per row of the U2 table (odd: rows in different banks)
  constexpr int RMX = ep2_rows_max(NMX, ep2_wide(sizeof(T), NB2, PRE));
  constexpr int UPL = PRE ? 1 : (NWX * NB2 * RMX + 63) / 64;  // U2 entries per lane
  const int nLinesYZ = p.m1 * p.m2;
  const int nTilesTot = p.nPanels * nLinesYZ;
  const int bid = blockIdx.x;
  const int perXcd = gridDim.x / 8;
  const int Lx = (bid % 8) * perXcd + bid / 8;
  if (Lx >= nTilesTot) return;
  const int yz = Lx / p.nPanels, panel = Lx % p.nPanels;
  const int slot = panel * nLinesYZ + yz;
  const int jy = yz % p.m1, jz = yz / p.m1;
  const int t = threadIdx.x;
  if (p.gate && *p.gate == 0) return;
  if (p.slotOn && !p.slotOn[slot]) {
    if (p.slotZero && t < kGMax * kCMax) p.partial[size_t(slot) * kGMax * kCMax + t] = 0.;
    return;
  }
  const unsigned long long mask = p.keepMask[slot];
  if (mask == 0ull) {
    if (t < kGMax * kCMax) p.partial[size_t(slot) * kGMax * kCMax + t] = 0.;
    return;
  }
  const int nm = ep2_exact(NMX) ? NMX : p.nm, nw = p.nw, ncol = nm * nw, R = p.rpw;
  const int kk = p.panelKK[panel];
  const int gstart = p.panelGStart[panel], gsize = __builtin_amdgcn_readfirstlane(p.panelGSize[panel]);
  const int is1 = p.kkStateOff[kk] + gstart;
  const double scrW = p.screen > 0. ? (p.screenOf ? p.screenOf[is1] : p.screen) : 0.;
  const double inv_g = 1. / double(float(gsize));
  // LDS: rows (64) | U2 (R x U2S double2) | g' (R x (NMX NB2 + 1) double2, zero beyond nm) | |g|^2 (R x NMX x
  //      NB2) | e2 (R x NB2) | occupations (CM x R x NB2) | e1 (kGMax) | ADAPT: widths (gsize x R x NB2)
  EpRow* rows = reinterpret_cast<EpRow*>(smem);
  double2* sU2 = reinterpret_cast<double2*>(rows + 64);
  constexpr int GPS = NMX * NB2 + 1;
  double2* gp = sU2 + (PRE ? 0 : size_t(R) * U2S);
  double* gsq = reinterpret_cast<double*>(gp + size_t(R) * GPS);
  double* se2 = gsq + size_t(R) * NMX * NB2;
  double* sf2 = se2 + R * NB2;
  double* se1 = sf2 + CM * R * NB2;
  double* sSig = se1 + kGMax;
  if (t < gsize) se1[t] = p.e1pool[is1 + t];
  for (int i = t; i < R * GPS; i += 64) gp[i] = make_double2(0., 0.);
  const int nkeep = __popcll(mask);
  {
    // q = k2 - k1 folded: its y and z are the slot's, x the row's
    int x1, y1, z1;
    mesh_coords(__builtin_amdgcn_readfirstlane(p.kkMesh[kk]), p.m0, p.m1, x1, y1, z1);
    const int dy = jy - y1 + (jy < y1 ? p.m1 : 0), dz = jz - z1 + (jz < z1 ? p.m2 : 0);
    const bool keep = t < p.m0 && ((mask >> t) & 1ull);
    int4 mr = make_int4(0, 0, 0, 0);
    if (keep) mr = p.meshRow[(jz * p.m1 + jy) * p.m0 + t];
    // the rows in order of their band counts, most first: a pass runs its largest
    // count for all of its rows, so rows of like counts share passes
    const unsigned long long below = (1ull << t) - 1ull;
    int pos = 0;
#pragma unroll
    for (int n = NB2; n >= 1; --n) {
      const unsigned long long same = __ballot(keep && mr.y == n);
      if (mr.y == n) pos += __popcll(same & below);
      else if (mr.y < n) pos += __popcll(same);
    }
    if (keep) rows[pos] = EpRow{t | mr.y << 8, (dz * p.m1 + dy) * p.m0 + t - x1 + (t < x1 ? p.m0 : 0), mr.z, mr.w};
  }
  __syncthreads();
  if (t == 0) {
    if (p.keptRows) atomicAdd(p.keptRows, (unsigned long long)nkeep);
    if (p.keptBands) {
      unsigned long long nb = 0;
      for (int i = 0; i < nkeep; ++i) nb += rows[i].jxnb >> 8;
      atomicAdd(p.keptBands, nb);
    }
  }
  // lane (r, sub): r < R rows of a pass, whole rows of nm lanes; the rest repeat row 0's first mode
  const bool laneOn = t < R * nm;
  const int r = laneOn ? t / nm : 0, sub = laneOn ? t - r * nm : 0;
  const T2v* G3 = static_cast<const T2v*>(p.G3) + size_t(slot) * p.m0 * ncol;
  const int rowG = p.nb2max * nm;  // PRE: g' row length, (b2, nu)
  const double2* GP = static_cast<const double2*>(p.G3) + size_t(slot) * p.m0 * rowG;
  const T2v* E3T = static_cast<const T2v*>(p.E3T);
  double part[GM][CM];
#pragma unroll
  for (int gi = 0; gi < GM; ++gi)
#pragma unroll
    for (int c = 0; c < CM; ++c) part[gi][c] = 0.;

  T2v g[PRE ? 1 : NWX];         // g3(nu = sub, w2) of the lane's row
  double2 gv[PRE ? NB2 : 1];    // PRE: g'(nu = sub, b2) of the lane's row
  T2v e3c[NMX];                 // e3(nu, nu2 = sub) at the row's q
  double2 u2v[UPL];             // U2 entries of the pass (lane-strided over R x NWX x NB2)
  double e2v = 0., f2v[CM], w3 = 0., n3[CM];
  int grp = 0;
  auto row_of = [&](int m0r, int rr) { return rows[min(m0r + rr, nkeep - 1)]; };
  auto load_g = [&](int m0r) {
    const EpRow ri = row_of(m0r, r);
    const int jx = ri.jxnb & 0xff;
    if constexpr (PRE) {
#pragma unroll
      for (int b2 = 0; b2 < NB2; ++b2) gv[b2] = GP[size_t(jx) * rowG + min(b2, (ri.jxnb >> 8) - 1) * nm + sub];
    } else {
      // a row's modes are neighbours, so one load's lanes fall into a few lines
      // (with w2 fastest every lane was in a line of its own); the w2 offset is
      // uniform, the lane's 32-bit offset the same for all of them
      const unsigned off = unsigned(jx * ncol + sub) * unsigned(sizeof(T2v));
#pragma unroll
      for (int w2 = 0; w2 < NWX; ++w2)
        g[w2] = *reinterpret_cast<const T2v*>(reinterpret_cast<const char*>(G3 + min(w2, nw - 1) * nm) + off);
    }
  };
  // U2 of the pass: entry i = (row, b2, w2), w2 fastest, NWX x NB2 per row; and the band
  // energies and occupations, lane = (row, b2) for lanes < R NB2
  auto load_u2 = [&](int m0r) {
    if constexpr (!PRE) {
#pragma unroll
      for (int u = 0; u < UPL; ++u) {  // NWX NB2 is one or two waves of entries: a row per load
        const EpRow q = row_of(m0r, min(64 * u / (NWX * NB2), R - 1));
        const int b2 = (t + 64 * u) % (NWX * NB2) / NWX, nb = __builtin_amdgcn_readfirstlane(q.jxnb >> 8);
        const double2* src = p.U2pool + __builtin_amdgcn_readfirstlane(q.u2off);
        const unsigned off = unsigned(min(b2, nb - 1) * nw + min(t % NWX, nw - 1)) * unsigned(sizeof(double2));
        u2v[u] = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(src) + off);
      }
    }
    const EpRow q = row_of(m0r, min(t / NB2, R - 1));
    const int st = q.soff + min(t % NB2, (q.jxnb >> 8) - 1);
    e2v = p.e2pool[st];
#pragma unroll
    for (int c = 0; c < CM; ++c) f2v[c] = p.fermi[size_t(min(c, p.nCalc - 1)) * p.numStates + st];
  };
  auto load_e3 = [&](int m0r) {
    const int iq = row_of(m0r, r).iq;
    // opaque: the offsets of the modes are worked out for each pass on the scalar
    // unit, not kept (and spilled) across the passes
    int st = nm;
    asm volatile("" : "+s"(st));
    const T2v* e3 = E3T + size_t(iq) * nm * nm + sub;
#pragma unroll
    for (int nu = 0; nu < NMX; ++nu) e3c[nu] = ep2_exact(NMX) ? e3[nu * NMX] : e3[min(nu, st - 1) * st];
    w3 = p.Wpool[size_t(iq) * nm + sub];
    grp = p.qModeGrp[size_t(iq) * nm + sub];
#pragma unroll
    for (int c = 0; c < CM; ++c) n3[c] = p.bose[(size_t(iq) * nm + sub) * p.nCalc + min(c, p.nCalc - 1)];
  };
  load_g(0);
  load_u2(0);
  load_e3(0);
  for (int m0r = 0; m0r < nkeep; m0r += R) {
    const int nr = min(R, nkeep - m0r);
    const bool rowOn = laneOn && r < nr;
    const EpRow ri = row_of(m0r, r);
    const int nb2 = rowOn ? ri.jxnb >> 8 : 0;
    // largest band count of the pass's rows
    int nbw = 1;
#pragma unroll
    for (int b = 1; b < NB2; ++b) nbw += __ballot(nb2 > b) != 0ull;
    // row data of the pass into LDS
    if constexpr (!PRE) {
#pragma unroll
      for (int u = 0; u < UPL; ++u) {
        const int rr = 64 * u / (NWX * NB2);
        if (rr < R) sU2[rr * U2S + (t + 64 * u) % (NWX * NB2)] = t % NWX < nw ? u2v[u] : make_double2(0., 0.);
      }
    }
    if (t < R * NB2) {
      se2[t] = e2v;
#pragma unroll
      for (int c = 0; c < CM; ++c) sf2[c * R * NB2 + t] = f2v[c];
      if constexpr (ADAPT) {
        // width of (b1 group member, row, b2): the lanes of a row share it
        const int rr = t / NB2;
        const EpRow q = row_of(m0r, rr);
        const int st = q.soff + min(t % NB2, (q.jxnb >> 8) - 1);
        for (int gi = 0; gi < gsize; ++gi) {
          double v[3], s = 0.;
          for (int d = 0; d < 3; ++d) v[d] = p.stateV[3 * (is1 + gi) + d] - p.stateV[3 * st + d];
          for (int d = 0; d < 3; ++d) {
            const double x = p.qT[3 * d] * v[0] + p.qT[3 * d + 1] * v[1] + p.qT[3 * d + 2] * v[2];
            s += x * x;
          }
          s = sqrt(s / 6.);
          if (s != 0. && s < p.minWidth) s = p.minWidth;
          if (v[0] == 0. && v[1] == 0. && v[2] == 0.) s = -1.;
          sSig[gi * R * NB2 + t] = s;
        }
      }
    }
    wave_sync();
    // A: electron rotation, thread nu = sub (PRE: done by the x-stage kernel)
    double2* out = gp + r * GPS + sub * NB2;
    if constexpr (PRE) {
      if (rowOn) {
#pragma unroll
        for (int b2 = 0; b2 < NB2; ++b2) out[b2] = gv[b2];
      }
    } else if (rowOn) {
      const double2* u = sU2 + r * U2S;
      int b = 0;
      for (; b + 1 < nbw; b += 2) ep2_rot_el<T2v, NWX, 2>(g, u + b * NWX, out + b);
      if (b < nbw) ep2_rot_el<T2v, NWX, 1>(g, u + b * NWX, out + b);
    }
    load_g(m0r + R);
    load_u2(m0r + R);
    wave_sync();
    // B: phonon rotation, thread nu2 = sub, then |g|^2 and the b2 groups
    double* gq = gsq + (r * NMX + sub) * NB2;
    if (rowOn) {
      const double2* x = gp + r * GPS;
      int b = 0;
      for (; b + 1 < nbw; b += 2) ep2_rot_ph<T2v, NMX, NB2, 2>(e3c, x + b, gq + b);
      if (b < nbw) ep2_rot_ph<T2v, NMX, NB2, 1>(e3c, x + b, gq + b);
    }
    const double w3c = w3;
    const int grpc = grp;
    double n3c[CM];
#pragma unroll
    for (int c = 0; c < CM; ++c) n3c[c] = n3[c];
    load_e3(m0r + R);
    if (rowOn) {
      const double* e2r = se2 + r * NB2;
      for (int b = 0; b < nb2;) {
        int deg = 0;
        for (int i = b; i < nb2; ++i) {
          if (fabs(e2r[b] - e2r[i]) < 1.0e-6) deg++;
          else break;
        }
        if (deg > 1) {
          double s2 = 0.;
          for (int i = 0; i < deg; ++i) s2 += gq[b + i] / double(float(deg));
          for (int i = 0; i < deg; ++i) gq[b + i] = s2;
        }
        b += deg;
      }
    }
    wave_sync();
    // C: the nu groups and the smearing weights
    if (rowOn && w3c >= p.cutoff) {
      const int mystart = grpc & 0xff, mydeg = grpc >> 8;
      const double* g0 = gsq + (r * NMX + mystart) * NB2;
      const double wfac = p.norm / w3c * 3.14159265358979323846;  // once per lane, not per term
#pragma unroll 1
      for (int b2 = 0; b2 < nb2; ++b2) {
        double vb;
        if (mydeg > 1) {
          vb = 0.;
          for (int i = 0; i < mydeg; ++i) vb += g0[i * NB2 + b2] / double(float(mydeg));
        } else {
          vb = gq[b2];
        }
        const double en2 = se2[r * NB2 + b2];
        const double cpl = vb * inv_g;
#pragma unroll
        for (int gi = 0; gi < GM; ++gi) {
          if (gi >= gsize) break;
          const double x1 = se1[gi] - en2 + w3c, x2 = se1[gi] - en2 - w3c;
          double d1, d2;
          if constexpr (ADAPT) {
            const AdaptiveWidth aw{sSig[gi * R * NB2 + r * NB2 + b2]};
            d1 = adaptive_delta(x1, aw);
            d2 = adaptive_delta(x2, aw);
          } else {
            if (p.screen > 0. && fmin(fabs(x1), fabs(x2)) * p.invSigma >= scrW) continue;
            d1 = gaussian_delta(x1, p.invSigma, p.deltaPref);
            d2 = gaussian_delta(x2, p.invSigma, p.deltaPref);
          }
          if (d1 <= 0. && d2 <= 0.) continue;
#pragma unroll
          for (int c = 0; c < CM; ++c) {
            if (c >= p.nCalc) break;
            const double f2 = sf2[(c * R + r) * NB2 + b2];
            part[gi][c] += cpl * ((f2 + n3c[c]) * d1 + (1. - f2 + n3c[c]) * d2) * wfac;
          }
        }
      }
    }
    wave_sync();  // the next pass rewrites the row data
  }
  // wave reduction of the partial linewidths into partial[slot]
  double* red = reinterpret_cast<double*>(smem);
#pragma unroll
  for (int gi = 0; gi < GM; ++gi) {
    if (gi >= gsize) break;
#pragma unroll
    for (int c = 0; c < CM; ++c) {
      double v = part[gi][c];
      for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
      if (t == 0) red[gi * kCMax + c] = v;
    }
  }
  __syncthreads();
  if (t < kGMax * kCMax) {
    const int c = t % kCMax, gi = t / kCMax;
    p.partial[size_t(slot) * kGMax * kCMax + t] = (c < CM && gi < gsize) ? red[t] : 0.;
  }
}

inline size_t sep_ep2_lds_bytes(int nmx, int nb2, int cm, int gm, int rpw, bool pre, bool adaptive) {
  size_t b = 64 * sizeof(EpRow);
  if (!pre) b += size_t(rpw) * (16 * nb2 + 1) * sizeof(double2);    // U2
  b += size_t(rpw) * (nmx * nb2 + 1) * sizeof(double2);             // g'
  b += size_t(rpw) * nmx * nb2 * sizeof(double);                    // |g|^2
  b += size_t(rpw) * nb2 * sizeof(double) * (1 + cm);               // e2, occupations
  b += size_t(kGMax) * sizeof(double);                              // e1
  if (adaptive) b += size_t(gm) * rpw * nb2 * sizeof(double);       // widths
  return std::max(b, size_t(kGMax) * kCMax * sizeof(double)) + 64;
}

template <typename T>
void launch_ep2(EpParams q, int gsizeMax, int grid, bool pre, hipStream_t s) {
  const int gm = gsizeMax > 0 ? gsizeMax : kGMax;
  PHX_REQUIRE(gm <= kGMax && q.nb2max <= kSepNb2 && q.nm <= kSepNm && q.nCalc <= kCMax,
              "separable transform: epilogue sizes");
  PHX_REQUIRE(!pre || (sizeof(T) == 4 && q.nm <= 16 && !q.adaptive), "separable transform: rotated x-stage is FP32 only");
  auto go = [&](auto nmx, auto small, auto cmx, auto prec) {
    constexpr int NM = decltype(nmx)::value, NB = decltype(small)::value ? 4 : 8, CM = decltype(cmx)::value;
    constexpr bool PRE = decltype(prec)::value == 1, ADAPT = decltype(prec)::value == 2;
    constexpr int GM = NB == 4 ? 4 : kGMax;
    q.rpw = std::min(64 / q.nm, ep2_rows_max(NM, ep2_wide(sizeof(T), NB, PRE)));
    const size_t lds = sep_ep2_lds_bytes(NM, NB, CM, gm, q.rpw, PRE, ADAPT);
    PHX_REQUIRE(lds <= 160 * 1024, "separable transform: LDS budget exceeded");
    auto kern = k_sep_ep2<T, CM, NM, GM, NB, PRE, ADAPT>;
    PHX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64), lds, s, q);
  };
  auto calcs = [&](auto nmx, auto small, auto prec) {
    if (q.nCalc == 1) go(nmx, small, std::integral_constant<int, 1>{}, prec);
    else if (q.nCalc == 2) go(nmx, small, std::integral_constant<int, 2>{}, prec);
    else go(nmx, small, std::integral_constant<int, kCMax>{}, prec);
  };
  // small: at most 4 bands per inner point and 4 members per b1 group, held per lane
  const bool small = q.nb2max <= 4 && gm <= 4;
  auto kinds = [&](auto nmx, auto kind) {
    small ? calcs(nmx, std::true_type{}, kind) : calcs(nmx, std::false_type{}, kind);
  };
  auto sizes = [&](auto nmx) {
    if constexpr (sizeof(T) == 4 && decltype(nmx)::value <= 24 && decltype(nmx)::value != 18) {  // up to 16 modes
      if (pre) return kinds(nmx, std::integral_constant<int, 1>{});
    }
    q.adaptive ? kinds(nmx, std::integral_constant<int, 2>{}) : kinds(nmx, std::integral_constant<int, 0>{});
  };
  switch (q.nm) {
    case 3: sizes(std::integral_constant<int, 3>{}); break;
    case 6: sizes(std::integral_constant<int, 6>{}); break;
    case 9: sizes(std::integral_constant<int, 9>{}); break;
    case 12: sizes(std::integral_constant<int, 12>{}); break;
    case 15: sizes(std::integral_constant<int, 15>{}); break;
    case 18: sizes(std::integral_constant<int, 18>{}); break;
    default:
      if (q.nm <= 24) sizes(std::integral_constant<int, 24>{});
      else sizes(std::integral_constant<int, kSepNm>{});
  }
  PHX_HIP(hipGetLastError());
}

}  // namespace phx
