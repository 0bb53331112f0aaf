// Reduction half of the phonon-linewidth builder (phel.hip): parameters and launcher.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace phx {

constexpr int kPhelPoints = 32;  // outer points per launch at most

// One launch takes np outer points; i-th point: nb1[i] bands at e1[i].
struct PhelParams {
  int nq, np, nb2, nm, nCalc;
  int nb1[kPhelPoints], e1[kPhelPoints];  // e1: offset in E1 (and, times 3, in v1)
  double* g2;             // per (point, q3) a block of g2Stride, (b1, b2, nu) column-major inside
  size_t g2Stride;
  const double* E1;       // energies of the outer states
  const double* E2;       // band energies of the k2 points, nb2 per point
  const int* e2off;       // per (point, q3): offset of its k2 point's energies in E2
  const double* W3;       // nq x nm
  const double* F1;       // per point a block of f1Stride: nCalc x nb1 values f (1 - f) of the k1 states
  size_t f1Stride;
  const double* invT;     // nCalc
  double norm, cutoff, invSigma, deltaPref;
  int adaptive;           // width from v1 - v2 (AdaptiveGaussianDeltaFunction)
  const double* v1;       // outer states x 3
  const double* V2;       // nq x nb2 x 3
  double qT[9], minWidth;
  double* lw;             // nCalc x nq x nm
};

void launch_phel_reduce(const PhelParams& p, hipStream_t s);
void launch_phel_rows(int np, int nq, int nw, const int* kmesh, const int* qmesh, const int* ik, int* u2off, int* e2off,
                      hipStream_t s);
void launch_phel_flag_failures(int n, const int* info, int* flag, hipStream_t s);

}  // namespace phx
