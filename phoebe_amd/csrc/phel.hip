// Phonon linewidths from electron-phonon scattering on gfx950
// (PhElScatteringMatrix::builder, phel_scattering.cpp:43-363), the reduction
// half: for one outer electron point k1 and all phonon wavevectors q3 of the
// mesh, the couplings |g(b1, b2, nu)|^2 at k2 = k1 + q3 (calcCouplingSquared in
// store mode, (b1, b2, nu) column-major per q3) are
//   * symmetrized over degenerate b1, then b2, then nu groups
//     (ScatteringMatrix::symmetrizeCoupling, scattering.cpp:1209-1318), and
//   * reduced into the phonon linewidths
//     Gamma(c, q3, nu) += sum_{b1, b2} |g|^2 F_c(b1) delta(e1 - e2 + w) norm / T_c * pi
//     with F = f (1 - f) = 1 / (4 cosh^2((e - mu) / 2T)) (phel_scattering.cpp:284-324).
// Every (q3, nu, c) entry is owned by one thread, which takes a launch's outer
// points in order and adds each one's term, so the sums are deterministic and do
// not depend on how the points are split into launches.
#include "coupling_kernel.hpp"
#include "phel.hpp"
#include "phx_common.hpp"

namespace phx {


// Grid (q3 blocks, outer points).
__global__ void __launch_bounds__(64) k_phel_sym(PhelParams p) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x, pt = blockIdx.y;
  if (q >= p.nq) return;
  const int nb1 = p.nb1[pt], nb2 = p.nb2, nm = p.nm;
  double* c = p.g2 + (size_t(pt) * p.nq + q) * p.g2Stride;
  auto C = [&](int a, int b, int v) -> double& { return c[a + size_t(nb1) * (b + size_t(nb2) * v)]; };
  const double* e1 = p.E1 + p.e1[pt];
  const double* e2 = p.E2 + p.e2off[size_t(pt) * p.nq + q];
  const double* w3 = p.W3 + size_t(q) * nm;
  for (int a = 0; a < nb1;) {
    int deg = 0;
    for (int i = a; i < nb1; ++i) {
      if (fabs(e1[a] - e1[i]) < 1.0e-6) ++deg;
      else break;
    }
    if (deg > 1)
      for (int b = 0; b < nb2; ++b)
        for (int v = 0; v < nm; ++v) {
          double s = 0.;
          for (int i = 0; i < deg; ++i) s += C(a + i, b, v) / double(float(deg));
          for (int i = 0; i < deg; ++i) C(a + i, b, v) = s;
        }
    a += deg;
  }
  for (int b = 0; b < nb2;) {
    int deg = 0;
    for (int i = b; i < nb2; ++i) {
      if (fabs(e2[b] - e2[i]) < 1.0e-6) ++deg;
      else break;
    }
    if (deg > 1)
      for (int a = 0; a < nb1; ++a)
        for (int v = 0; v < nm; ++v) {
          double s = 0.;
          for (int i = 0; i < deg; ++i) s += C(a, b + i, v) / double(float(deg));
          for (int i = 0; i < deg; ++i) C(a, b + i, v) = s;
        }
    b += deg;
  }
  for (int v = 0; v < nm;) {
    int deg = 0;
    for (int i = v; i < nm; ++i) {
      if (fabs(w3[v] - w3[i]) < 1.0e-6) ++deg;
      else break;
    }
    if (deg > 1)
      for (int a = 0; a < nb1; ++a)
        for (int b = 0; b < nb2; ++b) {
          double s = 0.;
          for (int i = 0; i < deg; ++i) s += C(a, b, v + i) / double(float(deg));
          for (int i = 0; i < deg; ++i) C(a, b, v + i) = s;
        }
    v += deg;
  }
}

__device__ inline double phel_delta(const PhelParams& p, const double* v1, double energy, int q, int b) {
  if (!p.adaptive) return gaussian_delta(energy, p.invSigma, p.deltaPref);
  const double* y = p.V2 + (size_t(q) * p.nb2 + b) * 3;
  const double d0 = v1[0] - y[0], d1 = v1[1] - y[1], d2 = v1[2] - y[2];
  if (d0 == 0. && d1 == 0. && d2 == 0.) return energy == 0. ? 1. : 0.;
  double s = 0.;
  for (int i = 0; i < 3; ++i) {
    const double d = p.qT[3 * i] * d0 + p.qT[3 * i + 1] * d1 + p.qT[3 * i + 2] * d2;
    s += d * d;
  }
  s = sqrt(s / 6.);
  if (s == 0.) return 0.;
  if (s < p.minWidth) s = p.minWidth;
  if (fabs(energy) > 2. * s) return 0.;
  const double t = energy / s;
  if (t > 6.) return 0.;
  return exp(-t * t) / 1.7724538509055160273 / s / 0.9953222650189527;
}

__global__ void __launch_bounds__(256) k_phel_rates(PhelParams p) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= p.nq * p.nm) return;
  const int q = t / p.nm, v = t % p.nm;
  const double w = p.W3[size_t(q) * p.nm + v];
  if (w < p.cutoff) return;  // phel_scattering.cpp:266-270
  const int nb2 = p.nb2;
  double sum[kCMax];
  for (int k = 0; k < kCMax; ++k) sum[k] = k < p.nCalc ? p.lw[(size_t(k) * p.nq + q) * p.nm + v] : 0.;
  for (int pt = 0; pt < p.np; ++pt) {
    const int nb1 = p.nb1[pt];
    const double* c = p.g2 + (size_t(pt) * p.nq + q) * p.g2Stride;
    const double* e1 = p.E1 + p.e1[pt];
    const double* e2 = p.E2 + p.e2off[size_t(pt) * p.nq + q];
    const double* F1 = p.F1 + pt * p.f1Stride;
    double acc[kCMax];
    for (int k = 0; k < kCMax; ++k) acc[k] = 0.;
    for (int a = 0; a < nb1; ++a)
      for (int b = 0; b < nb2; ++b) {
        const double d = phel_delta(p, p.v1 + 3 * size_t(p.e1[pt] + a), e1[a] - e2[b] + w, q, b);
        if (!(d > 0.)) continue;
        const double g = c[a + size_t(nb1) * (b + size_t(nb2) * v)];
        for (int k = 0; k < kCMax; ++k)
          if (k < p.nCalc) acc[k] += g * F1[size_t(k) * nb1 + a] * d * p.norm * p.invT[k] * 3.14159265358979323846;
      }
    for (int k = 0; k < kCMax; ++k) sum[k] += acc[k];
  }
  for (int k = 0; k < kCMax; ++k)
    if (k < p.nCalc) p.lw[(size_t(k) * p.nq + q) * p.nm + v] = sum[k];
}

// Rows of np outer points on the k mesh: for point i (mesh index ik[i]) and q3 of
// the q mesh, which divides the k mesh, k2 = k1 + q3 (first index fastest): its
// eigenvectors at u2off, its energies at e2off.
__global__ void __launch_bounds__(256) k_phel_rows(int nq, int nw, int3 km, int3 qm, const int* __restrict__ ik,
                                                   int* __restrict__ u2off, int* __restrict__ e2off) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y;
  if (q >= nq) return;
  int x, y, z, qx, qy, qz;
  mesh_coords(ik[i], km.x, km.y, x, y, z);
  mesh_coords(q, qm.x, qm.y, qx, qy, qz);
  x = (x + qx * (km.x / qm.x)) % km.x;
  y = (y + qy * (km.y / qm.y)) % km.y;
  z = (z + qz * (km.z / qm.z)) % km.z;
  const int k = (z * km.y + y) * km.x + x;
  u2off[size_t(i) * nq + q] = k * nw * nw;
  e2off[size_t(i) * nq + q] = k * nw;
}

void launch_phel_rows(int np, int nq, int nw, const int* kmesh, const int* qmesh, const int* ik, int* u2off, int* e2off,
                      hipStream_t s) {
  if (np <= 0 || nq <= 0) return;
  hipLaunchKernelGGL(k_phel_rows, dim3(ceil_div(nq, 256), np), dim3(256), 0, s, nq, nw,
                     make_int3(kmesh[0], kmesh[1], kmesh[2]), make_int3(qmesh[0], qmesh[1], qmesh[2]), ik, u2off, e2off);
  PHX_HIP(hipGetLastError());
}

// flag[0] = 1 when any eigensolve status in info[0..n) is negative
__global__ void __launch_bounds__(256) k_phel_flag_failures(int n, const int* info, int* flag) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && info[i] < 0) flag[0] = 1;
}

void launch_phel_flag_failures(int n, const int* info, int* flag, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_phel_flag_failures, dim3(ceil_div(n, 256)), dim3(256), 0, s, n, info, flag);
  PHX_HIP(hipGetLastError());
}

void launch_phel_reduce(const PhelParams& p, hipStream_t s) {
  if (p.nq <= 0 || p.np <= 0) return;
  if (p.np > kPhelPoints) throw Error(-1, "ph-el linewidths: too many outer points per launch");
  if (p.nCalc < 1 || p.nCalc > kCMax) throw Error(-1, "ph-el linewidths: 1..4 (T, mu) calculations");
  hipLaunchKernelGGL(k_phel_sym, dim3(ceil_div(p.nq, 64), p.np), dim3(64), 0, s, p);
  PHX_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_phel_rates, dim3(ceil_div((long long)p.nq * p.nm, 256)), dim3(256), 0, s, p);
  PHX_HIP(hipGetLastError());
}

}  // namespace phx
