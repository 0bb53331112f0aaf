// Batched Hermitian eigensolver, LDS resident.
//
// Replaces kokkosZHEEV (common_kokkos.cpp:11-100): eigenvalues ascending,
// eigenvectors written over the input as the columns of a column-major
// matrix (each matrix contiguous, LayoutStride (N^2,1,N), common_kokkos.cpp:
// 32-41; electron_h0_wannier.cpp:787-791).  Electrons: k_eig_ql.  Phonons: a
// parallel cyclic complex Jacobi method with round-robin pair ordering: all N/2
// disjoint rotations of a round are applied at once, the matrix and the
// accumulated eigenvectors stay in LDS for all sweeps.
//
// The phonon kernels fuse the steps either side of the eigensolve in
// PhononH0::kokkosBatchedBuildBlochHamiltonian / DiagonalizeFromCoordinates
// (phonon_h0_kokkos.cpp:150-170, 186-219): D <- (D + D^H)/2 / sqrt(M_m M_n)
// before, omega = sign(l) sqrt|l| and e_m <- e_m / sqrt(M_m) after.
#include "phx_common.hpp"

namespace phx {

__device__ inline double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ inline double2 cconj(double2 a) { return make_double2(a.x, -a.y); }

// One rotation of a round: J = [[c, s e^{i phi}], [-s e^{-i phi}, c]] on (p, q).
struct Rot {
  int p, q;
  double c;
  double2 sp;  // s e^{+i phi}
  double2 sm;  // s e^{-i phi}
};

__device__ inline int rr_player(int pos, int round, int n) {
  // circle method: player 0 fixed, the others rotate by one per round
  if (pos == 0) return 0;
  return (round + pos - 1) % (n - 1) + 1;
}

__global__ void __launch_bounds__(64) k_jacobi(int N, int M, double2* __restrict__ A,
                                               double* __restrict__ W, int* __restrict__ info,
                                               const double* __restrict__ masses, int maxSweeps) {
  extern __shared__ double2 lds[];
  const int mat = blockIdx.x;
  if (mat >= M) return;
  const int lane = threadIdx.x;
  const int NN = N * N;
  double2* a = lds;
  double2* v = lds + NN;
  Rot* rot = reinterpret_cast<Rot*>(v + NN);
  double* red = reinterpret_cast<double*>(rot + 32);
  double2* Am = A + size_t(mat) * NN;

  // load (column-major) with hermitization
  for (int e = lane; e < NN; e += 64) {
    int i = e % N, j = e / N;
    double2 x;
    double2 aij = Am[i + N * j], aji = Am[j + N * i];
    x = make_double2(0.5 * (aij.x + aji.x), 0.5 * (aij.y - aji.y));
    x.x /= sqrt(masses[i] * masses[j]);
    x.y /= sqrt(masses[i] * masses[j]);
    a[e] = x;
    v[e] = make_double2(i == j ? 1. : 0., 0.);
  }
  __syncthreads();

  double part = 0.;
  for (int e = lane; e < NN; e += 64) part += a[e].x * a[e].x + a[e].y * a[e].y;
  for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o);
  const double norm2 = part;

  const int n = N + (N & 1);  // even number of players (N is a dummy when odd)
  const int npairs = n / 2;
  int sweep = 0;
  bool converged = false;
  for (; sweep < maxSweeps; ++sweep) {
    double off = 0.;
    for (int e = lane; e < NN; e += 64) {
      int i = e % N, j = e / N;
      if (i != j) off += a[e].x * a[e].x + a[e].y * a[e].y;
    }
    for (int o = 32; o > 0; o >>= 1) off += __shfl_xor(off, o);
    if (off <= 1e-30 * norm2) {
      converged = true;
      break;
    }
    for (int r = 0; r < n - 1; ++r) {
      if (lane < npairs) {
        int p = rr_player(lane, r, n), q = rr_player(n - 1 - lane, r, n);
        if (p > q) { int t = p; p = q; q = t; }
        Rot R;
        R.p = p;
        R.q = q;
        R.c = 1.;
        R.sp = make_double2(0., 0.);
        R.sm = make_double2(0., 0.);
        if (q < N) {
          double2 apq = a[p + N * q];
          double rr = sqrt(apq.x * apq.x + apq.y * apq.y);
          if (rr > 1e-300) {
            double app = a[p + N * p].x, aqq = a[q + N * q].x;
            double tau = (aqq - app) / (2. * rr);
            double t = (tau >= 0. ? 1. : -1.) / (fabs(tau) + sqrt(1. + tau * tau));
            double c = 1. / sqrt(1. + t * t);
            double s = t * c;
            double2 ph = make_double2(apq.x / rr, apq.y / rr);
            R.c = c;
            R.sp = make_double2(s * ph.x, s * ph.y);
            R.sm = make_double2(s * ph.x, -s * ph.y);
          } else {
            R.q = N;  // nothing to do
          }
        }
        rot[lane] = R;
      }
      __syncthreads();
      // A <- A J and V <- V J (columns p, q of every pair)
      for (int it = lane; it < N * npairs; it += 64) {
        int k = it % N, pr = it / N;
        Rot R = rot[pr];
        if (R.q >= N) continue;
        double2 akp = a[k + N * R.p], akq = a[k + N * R.q];
        double2 t1 = cmul(akq, R.sm), t2 = cmul(akp, R.sp);
        a[k + N * R.p] = make_double2(akp.x * R.c - t1.x, akp.y * R.c - t1.y);
        a[k + N * R.q] = make_double2(t2.x + akq.x * R.c, t2.y + akq.y * R.c);
        double2 vkp = v[k + N * R.p], vkq = v[k + N * R.q];
        t1 = cmul(vkq, R.sm);
        t2 = cmul(vkp, R.sp);
        v[k + N * R.p] = make_double2(vkp.x * R.c - t1.x, vkp.y * R.c - t1.y);
        v[k + N * R.q] = make_double2(t2.x + vkq.x * R.c, t2.y + vkq.y * R.c);
      }
      __syncthreads();
      // A <- J^H A (rows p, q of every pair)
      for (int it = lane; it < N * npairs; it += 64) {
        int k = it % N, pr = it / N;
        Rot R = rot[pr];
        if (R.q >= N) continue;
        double2 apk = a[R.p + N * k], aqk = a[R.q + N * k];
        double2 t1 = cmul(R.sp, aqk), t2 = cmul(R.sm, apk);
        a[R.p + N * k] = make_double2(R.c * apk.x - t1.x, R.c * apk.y - t1.y);
        a[R.q + N * k] = make_double2(t2.x + R.c * aqk.x, t2.y + R.c * aqk.y);
      }
      __syncthreads();
      if (lane < npairs) {
        Rot R = rot[lane];
        if (R.q < N) {
          a[R.p + N * R.q] = make_double2(0., 0.);
          a[R.q + N * R.p] = make_double2(0., 0.);
          a[R.p + N * R.p].y = 0.;
          a[R.q + N * R.q].y = 0.;
        }
      }
      __syncthreads();
    }
  }
  // ascending order by rank (stable)
  if (lane < N) red[lane] = a[lane + N * lane].x;
  __syncthreads();
  for (int i = lane; i < N; i += 64) {
    double di = red[i];
    int rank = 0;
    for (int j = 0; j < N; ++j) {
      double dj = red[j];
      rank += (dj < di) || (dj == di && j < i);
    }
    double lam = di;
    lam = lam > 0. ? sqrt(lam) : -sqrt(-lam);
    W[size_t(mat) * N + rank] = lam;
    for (int k = 0; k < N; ++k) {
      double2 x = v[k + N * i];
      double s = sqrt(masses[k]);
      x.x /= s;
      x.y /= s;
      Am[k + N * rank] = x;
    }
  }
  if (lane == 0 && info) info[mat] = converged ? sweep : -1;
}

size_t jacobi_lds_bytes(int N) {
  return size_t(2) * N * N * sizeof(double2) + 32 * sizeof(Rot) + 64 * sizeof(double);
}

// The Jacobi method with the order N fixed at compile time and 64 / L
// matrices per wavefront, L >= N lanes each: every lane works on one matrix,
// index arithmetic is by constants, and a wave issues its instructions for
// several matrices at once.  Each matrix goes through the rotations of the
// one-matrix kernel, in the same order, with the same arithmetic per
// element; the wave runs sweeps until all its matrices have converged (a
// converged matrix's rotations are skipped, so its result and sweep count
// are its own).
template <int N, int L>
__global__ void __launch_bounds__(64) k_jacobi_n(int M, double2* __restrict__ A, double* __restrict__ W,
                                                 int* __restrict__ info, const double* __restrict__ masses,
                                                 int maxSweeps) {
  constexpr int G = 64 / L, NN = N * N, NE = N + (N & 1), NP = NE / 2;
  static_assert(L >= N && 64 % L == 0, "a matrix needs at least N lanes");
  extern __shared__ double2 lds[];
  const int lane = threadIdx.x, sg = lane / L, li = lane % L;
  const int mat = blockIdx.x * G + sg;
  const bool on = mat < M;
  double2* a = lds + size_t(sg) * 2 * NN;
  double2* v = a + NN;
  Rot* rot = reinterpret_cast<Rot*>(lds + size_t(G) * 2 * NN) + sg * NP;
  double* red = reinterpret_cast<double*>(reinterpret_cast<Rot*>(lds + size_t(G) * 2 * NN) + G * NP) + sg * N;
  double2* Am = A + size_t(on ? mat : 0) * NN;

  for (int e = li; e < NN; e += L) {
    const int i = e % N, j = e / N;
    double2 x = make_double2(0., 0.);
    if (on) {
      const double2 aij = Am[i + N * j], aji = Am[j + N * i];
      x = make_double2(0.5 * (aij.x + aji.x), 0.5 * (aij.y - aji.y));
      x.x /= sqrt(masses[i] * masses[j]);
      x.y /= sqrt(masses[i] * masses[j]);
    }
    a[e] = x;
    v[e] = make_double2(i == j ? 1. : 0., 0.);
  }
  __syncthreads();
  double part = 0.;
  for (int e = li; e < NN; e += L) part += a[e].x * a[e].x + a[e].y * a[e].y;
  for (int o = L / 2; o > 0; o >>= 1) part += __shfl_xor(part, o);
  const double norm2 = part;

  int sweep = 0, mySweeps = -1;
  for (; sweep < maxSweeps; ++sweep) {
    double off = 0.;
    for (int e = li; e < NN; e += L) {
      const int i = e % N, j = e / N;
      if (i != j) off += a[e].x * a[e].x + a[e].y * a[e].y;
    }
    for (int o = L / 2; o > 0; o >>= 1) off += __shfl_xor(off, o);
    if (mySweeps < 0 && off <= 1e-30 * norm2) mySweeps = sweep;
    if (__all(mySweeps >= 0)) break;
    const bool active = mySweeps < 0;
    for (int r = 0; r < NE - 1; ++r) {
      if (li < NP) {
        int pp = rr_player(li, r, NE), qq = rr_player(NE - 1 - li, r, NE);
        if (pp > qq) { const int t = pp; pp = qq; qq = t; }
        Rot R;
        R.p = pp;
        R.q = qq;
        R.c = 1.;
        R.sp = make_double2(0., 0.);
        R.sm = make_double2(0., 0.);
        if (qq < N && active) {
          const double2 apq = a[pp + N * qq];
          const double rr = sqrt(apq.x * apq.x + apq.y * apq.y);
          if (rr > 1e-300) {
            const double app = a[pp + N * pp].x, aqq = a[qq + N * qq].x;
            const double tau = (aqq - app) / (2. * rr);
            const double t = (tau >= 0. ? 1. : -1.) / (fabs(tau) + sqrt(1. + tau * tau));
            const double c = 1. / sqrt(1. + t * t);
            const double sn = t * c;
            const double2 ph = make_double2(apq.x / rr, apq.y / rr);
            R.c = c;
            R.sp = make_double2(sn * ph.x, sn * ph.y);
            R.sm = make_double2(sn * ph.x, -sn * ph.y);
          } else {
            R.q = N;
          }
        } else {
          R.q = N;  // dummy player, or a converged matrix
        }
        rot[li] = R;
      }
      __syncthreads();
      // A <- A J and V <- V J (columns p, q of every pair)
      for (int it = li; it < N * NP; it += L) {
        const int k = it % N, pr = it / N;
        const Rot R = rot[pr];
        if (R.q >= N) continue;
        const double2 akp = a[k + N * R.p], akq = a[k + N * R.q];
        double2 t1 = cmul(akq, R.sm), t2 = cmul(akp, R.sp);
        a[k + N * R.p] = make_double2(akp.x * R.c - t1.x, akp.y * R.c - t1.y);
        a[k + N * R.q] = make_double2(t2.x + akq.x * R.c, t2.y + akq.y * R.c);
        const double2 vkp = v[k + N * R.p], vkq = v[k + N * R.q];
        t1 = cmul(vkq, R.sm);
        t2 = cmul(vkp, R.sp);
        v[k + N * R.p] = make_double2(vkp.x * R.c - t1.x, vkp.y * R.c - t1.y);
        v[k + N * R.q] = make_double2(t2.x + vkq.x * R.c, t2.y + vkq.y * R.c);
      }
      __syncthreads();
      // A <- J^H A (rows p, q of every pair)
      for (int it = li; it < N * NP; it += L) {
        const int k = it % N, pr = it / N;
        const Rot R = rot[pr];
        if (R.q >= N) continue;
        const double2 apk = a[R.p + N * k], aqk = a[R.q + N * k];
        const double2 t1 = cmul(R.sp, aqk), t2 = cmul(R.sm, apk);
        a[R.p + N * k] = make_double2(R.c * apk.x - t1.x, R.c * apk.y - t1.y);
        a[R.q + N * k] = make_double2(t2.x + R.c * aqk.x, t2.y + R.c * aqk.y);
      }
      __syncthreads();
      if (li < NP) {
        const Rot R = rot[li];
        if (R.q < N) {
          a[R.p + N * R.q] = make_double2(0., 0.);
          a[R.q + N * R.p] = make_double2(0., 0.);
          a[R.p + N * R.p].y = 0.;
          a[R.q + N * R.q].y = 0.;
        }
      }
      __syncthreads();
    }
  }
  // ascending order by rank (stable)
  if (li < N) red[li] = a[li + N * li].x;
  __syncthreads();
  if (on && li < N) {
    const int i = li;
    const double di = red[i];
    int rank = 0;
    for (int j = 0; j < N; ++j) {
      const double dj = red[j];
      rank += (dj < di) || (dj == di && j < i);
    }
    double lam = di;
    lam = lam > 0. ? sqrt(lam) : -sqrt(-lam);
    W[size_t(mat) * N + rank] = lam;
    for (int k = 0; k < N; ++k) {
      double2 x = v[k + N * i];
      const double s = sqrt(masses[k]);
      x.x /= s;
      x.y /= s;
      Am[k + N * rank] = x;
    }
  }
  if (on && li == 0 && info) info[mat] = mySweeps >= 0 ? mySweeps : -1;
}

// ------------------------------------------------------------------ tridiagonal form and QL
// Electron matrices, any order: Householder reduction to a real tridiagonal
// matrix, the unitary factor formed in place, and implicit QL iterations with
// Wilkinson's shift on it (Bowdler, Martin, Reinsch and Wilkinson, Numerische
// Mathematik 11 (1968) 293-306), about a tenth of the operations of cyclic
// Jacobi.  L lanes per matrix, L >= N the next of 8, 16, 32, 64, so 64 / L
// matrices per wave; the matrix, then the factor, is the only array in LDS
// (rows padded to an odd length, since both phases run through rows and through
// columns).  A lane is a row in the reduction and in the rotations, a column
// while the factor is formed; the scalar recurrences of QL are computed by all
// lanes of a group alike, and the groups of a wave go through their (matrix,
// eigenvalue, iteration) states in one loop, so a group never waits for
// another's eigenvalue.
// Bound by latency: the rotations' chain of dependent FP64 operations, at the
// seven waves per CU whose matrices fit LDS.  32768 matrices of order 16: 3.85 ms
// with one Jacobi matrix per wave (LDS-bound), 1.2 so.  The phonons keep Jacobi, which finds the small
// eigenvalues of D(q), whose square roots are the acoustic frequencies, to better
// than the norm's rounding.
__device__ __forceinline__ void group_sync() {  // orders a wave's LDS accesses
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// v of the lane that a DPP control names (within rows of 16 lanes)
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  union { double d; int i[2]; } x{v};
  x.i[0] = __builtin_amdgcn_update_dpp(0, x.i[0], CTRL, 0xf, 0xf, true);
  x.i[1] = __builtin_amdgcn_update_dpp(0, x.i[1], CTRL, 0xf, 0xf, true);
  return x.d;
}

// Sum over the L lanes of a group, the same in all of them: neighbours, quads
// and halves of a row by DPP, rows by shuffles.
template <int L>
__device__ __forceinline__ double group_sum(double v) {
  v += dpp_move<0xB1>(v);              // quad_perm [1, 0, 3, 2]
  v += dpp_move<0x4E>(v);              // quad_perm [2, 3, 0, 1]
  v += dpp_move<0x141>(v);             // row_half_mirror: the other quad of 8
  if (L >= 16) v += dpp_move<0x140>(v);  // row_mirror: the other 8 of 16
#pragma unroll
  for (int o = 16; o < L; o *= 2) v += __shfl_xor(v, o);
  return v;
}

// 1 / sqrt(x), x normal: the hardware estimate and one third-order step.
__device__ __forceinline__ double rsqrt_refined(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double h = fma(-x * y, y, 1.);
  return fma(y * h, fma(0.375, h, 0.5), y);
}

inline size_t ql_lds_bytes(int N, int L) {
  const size_t ld = N | 1;
  return size_t(64 / L) * ((size_t(N) * ld + 2 * N) * sizeof(double2) + (size_t(2) * N + 2) * sizeof(double));
}

// Below this an element next to a largest component near one counts as zero: far
// below the norm's rounding, and its square is a normal number.
constexpr double kQlTiny = 1e-140;
// QL iterations of a matrix of order N: at most 30 N, as two or three per eigenvalue
// are usual but one alone can take about N (rank one with structured phases).
constexpr int kQlMaxIter = 30;

template <int L>
__global__ void __launch_bounds__(64) k_eig_ql(int N, int M, double2* __restrict__ A, double* __restrict__ W,
                                               int* __restrict__ info) {
  extern __shared__ double2 lds[];
  const int lane = threadIdx.x, sg = lane / L, li = lane % L;
  const int mat = blockIdx.x * (64 / L) + sg;
  const bool on = mat < M;
  const int ld = N | 1;
  double2* a = lds + size_t(sg) * (size_t(N) * ld + 2 * N);  // (row, column) at row + ld column
  double2* sv = a + size_t(N) * ld;                          // Householder vector
  double2* sw = sv + N;
  double* d = reinterpret_cast<double*>(lds + size_t(64 / L) * (size_t(N) * ld + 2 * N)) + size_t(sg) * (2 * N + 2);
  double* e = d + N;
  double2* Am = A + size_t(on ? mat : 0) * N * N;
  const bool row = li < N;

  // the lower triangle is the reference (uplo = L); scaled by a power of two to
  // a largest component near one, so that no square overflows; what a square that
  // underflows can lose is below kQlTiny
  double big = 0.;
#pragma unroll 4
  for (int j = 0; j < N; ++j) {
    double2 x = make_double2(0., 0.);
    if (row && on) {
      x = li >= j ? Am[li + N * j] : cconj(Am[j + N * li]);
      if (li == j) x.y = 0.;
    }
    if (row) a[li + ld * j] = x;
    big = fmax(big, fmax(fabs(x.x), fabs(x.y)));
  }
#pragma unroll
  for (int o = L / 2; o > 0; o >>= 1) big = fmax(big, __shfl_xor(big, o));
  const int ex = big > 0. && big < HUGE_VAL ? ilogb(big) : 0;
  group_sync();
  if (row)
    for (int j = 0; j < N; ++j) {
      const double2 x = a[li + ld * j];
      a[li + ld * j] = make_double2(ldexp(x.x, -ex), ldexp(x.y, -ex));
    }
  group_sync();

  // Householder: reflector k = I - tau v v^H, v(k + 1) = 1, maps column k below the
  // diagonal to the real number beta; A <- H^H A H as A - v w^H - w v^H.
  // v stays in column k (rows > k + 1), tau in sw's place at the end: kept in e's lanes
  double2 tauK = make_double2(0., 0.);  // lane k holds tau of reflector k
  for (int k = 0; k + 1 < N; ++k) {
    const bool in = row && li > k;
    const double2 x = in ? a[li + ld * k] : make_double2(0., 0.);
    const double2 alpha = a[k + 1 + ld * k];
    const double tail = group_sum<L>(li > k + 1 ? x.x * x.x + x.y * x.y : 0.);
    const double norm2 = alpha.x * alpha.x + alpha.y * alpha.y + tail;
    double beta = alpha.x;
    double2 tau = make_double2(0., 0.), v = make_double2(li == k + 1 ? 1. : 0., 0.);
    if (norm2 < kQlTiny * kQlTiny) {  // the column counts as zero: its square is no longer exact, nor is 1 / square finite
      beta = 0.;
    } else if (tail > 0. || alpha.y != 0.) {
      beta = sqrt(norm2);
      if (alpha.x > 0.) beta = -beta;
      tau = make_double2((beta - alpha.x) / beta, -alpha.y / beta);
      // x / (alpha - beta)
      const double ar = alpha.x - beta, ai = alpha.y, q = 1. / (ar * ar + ai * ai);
      if (li > k + 1) v = make_double2((x.x * ar + x.y * ai) * q, (x.y * ar - x.x * ai) * q);
    }
    if (!in) v = make_double2(0., 0.);
    if (li == k) tauK = tau;
    if (li == 0) e[k] = beta;
    if (in) sv[li] = v;
    group_sync();
    // p = tau A v
    double2 p = make_double2(0., 0.);
    if (in)
#pragma unroll 4
      for (int j = k + 1; j < N; ++j) {
        const double2 aj = a[li + ld * j], vj = sv[j];
        p.x += aj.x * vj.x - aj.y * vj.y;
        p.y += aj.x * vj.y + aj.y * vj.x;
      }
    p = tau.x != 0. || tau.y != 0. ? cmul(tau, p) : make_double2(0., 0.);  // identity: infinities stay where they are
    // w = p - (tau / 2) (p^H v) v, with tau p^H v = |tau|^2 v^H A v real
    const double2 pv = make_double2(group_sum<L>(in ? p.x * v.x + p.y * v.y : 0.),
                                    group_sum<L>(in ? p.x * v.y - p.y * v.x : 0.));
    const double h = -0.5 * (tau.x * pv.x - tau.y * pv.y);
    const double2 w = make_double2(p.x + h * v.x, p.y + h * v.y);
    if (in) sw[li] = w;
    group_sync();
    if (in) {
#pragma unroll 4
      for (int j = k + 1; j < N; ++j) {
        const double2 vj = sv[j], wj = sw[j];
        double2 aj = a[li + ld * j];
        aj.x -= v.x * wj.x + v.y * wj.y + w.x * vj.x + w.y * vj.y;
        aj.y -= v.y * wj.x - v.x * wj.y + w.y * vj.x - w.x * vj.y;
        a[li + ld * j] = aj;
      }
      if (li > k + 1) a[li + ld * k] = v;
    }
    group_sync();
  }
  if (row) d[li] = a[li + ld * li].x;
  if (li == 0) e[N - 1] = 0.;

  // Q = H_0 H_1 ... H_{N-2} in place: column k + 1 from reflector k (in column k), the
  // columns beyond it (lane = column) by H_k
  for (int k = N - 2; k >= 0; --k) {
    const double2 tau = make_double2(__shfl(tauK.x, sg * L + k), __shfl(tauK.y, sg * L + k));
    if (li > k + 1 && row) {
      double2 y = make_double2(0., 0.);
#pragma unroll 4
      for (int i = k + 2; i < N; ++i) {
        const double2 v = a[i + ld * k], q = a[i + ld * li];
        y.x += v.x * q.x + v.y * q.y;
        y.y += v.x * q.y - v.y * q.x;
      }
      y = cmul(tau, y);
      a[k + 1 + ld * li] = make_double2(-y.x, -y.y);
#pragma unroll 4
      for (int i = k + 2; i < N; ++i) {
        const double2 v = a[i + ld * k];
        double2 q = a[i + ld * li];
        q.x -= v.x * y.x - v.y * y.y;
        q.y -= v.x * y.y + v.y * y.x;
        a[i + ld * li] = q;
      }
    }
    group_sync();
    if (li > k && row) {  // lane = row
      const double2 v = li == k + 1 ? make_double2(1., 0.) : a[li + ld * k];
      const double2 t = cmul(tau, v);
      a[li + ld * (k + 1)] = make_double2((li == k + 1 ? 1. : 0.) - t.x, -t.y);
    }
    group_sync();
  }
  if (row) {
    a[li] = make_double2(li == 0 ? 1. : 0., 0.);
    a[ld * li] = make_double2(li == 0 ? 1. : 0., 0.);
  }
  group_sync();

  const unsigned long long ones = L == 64 ? ~0ull : (1ull << (L & 63)) - 1ull;  // a group's lanes in a ballot
  // implicit QL: eigenvalue l of the group, it iterations spent on it
  int l = 0, it = 0, total = 0, worst = 0;
  bool bad = false;
  while (__any(l < N && !bad)) {
    if (l < N && !bad) {
      // the first negligible off-diagonal from l on ends the block l .. m
      bool small = false;
      if (li >= l && li < N - 1)
        small = fabs(e[li]) <= fmax(kQlTiny, 2.220446049250313e-16 * (fabs(d[li]) + fabs(d[li + 1])));
      const unsigned long long hit = (__ballot(small) >> (sg * L)) & ones;
      const int m = hit ? __ffsll(hit) - 1 : N - 1;
      if (m == l) {
        ++l;
        it = 0;
      } else if (total == kQlMaxIter * N) {
        bad = true;
      } else {
        ++it;
        ++total;
        worst = max(worst, it);
        const double dl = d[l], el = e[l];
        double g = (d[l + 1] - dl) / (2. * el);
        g = d[m] - dl + el / (g + copysign(sqrt(g * g + 1.), g));
        double s = 1., c = 1., p = 0.;
        double2 f2 = row ? a[li + ld * m] : make_double2(0., 0.);  // column i + 1 of the lane's row
        double dn = d[m];                                        // d(i + 1)
        double di = d[m - 1], ei = e[m - 1];
        double2 z = row ? a[li + ld * (m - 1)] : make_double2(0., 0.);
        int i = m - 1;
        bool cut = false;
        for (; i >= l; --i) {
          // the next rotation's operands, while this one's chain runs
          const int in = max(i - 1, 0);
          const double dnx = d[in], enx = e[in];
          const double2 znx = row ? a[li + ld * in] : make_double2(0., 0.);
          const double f = s * ei, b = c * ei;
          const double r2 = f * f + g * g;
          // zero next to the largest component, near one: the block splits at i + 1.  Never the first
          // rotation, where f = e(m - 1) > kQlTiny, so every iteration changes the matrix
          if (r2 < 1e-290) {
            if (li == 0) {
              e[i + 1] = 0.;
              d[i + 1] = dn - p;
              e[m] = 0.;
            }
            cut = true;
            break;
          }
          const double ri = rsqrt_refined(r2);
          if (li == 0) e[i + 1] = r2 * ri;
          s = f * ri;
          c = g * ri;
          g = dn - p;
          const double t = (di - g) * s + 2. * c * b;
          p = s * t;
          if (li == 0) d[i + 1] = g + p;
          g = c * t - b;
          // columns i, i + 1 of the eigenvectors
          if (row) a[li + ld * (i + 1)] = make_double2(s * z.x + c * f2.x, s * z.y + c * f2.y);
          f2 = make_double2(c * z.x - s * f2.x, c * z.y - s * f2.y);
          dn = di;
          di = dnx;
          ei = enx;
          z = znx;
        }
        if (row) a[li + ld * (i + 1)] = f2;
        if (!cut && li == 0) {
          d[l] = dn - p;
          e[l] = g;
          e[m] = 0.;
        }
      }
    }
    group_sync();
  }

  // a NaN on the diagonal alone passes every test above
  bad = bad || ((__ballot(row && d[li] != d[li]) >> (sg * L)) & ones) != 0ull;

  // ascending order by rank (stable); lane = eigenvalue, then lane = row
  int rank = 0;
  if (row) {
    const double di = d[li];
    for (int j = 0; j < N; ++j) {
      const double dj = d[j];
      rank += (dj < di) || (dj == di && j < li);
    }
    if (on) W[size_t(mat) * N + rank] = ldexp(di, ex);
  }
  for (int j = 0; j < N; ++j) {
    const int r = __shfl(rank, sg * L + j);
    if (row && on) Am[li + N * r] = a[li + ld * j];
  }
  if (on && li == 0 && info) info[mat] = bad ? -1 : worst;
}

template <int N, int L>
static size_t jacobi_n_lds_bytes() {
  constexpr int G = 64 / L, NE = N + (N & 1);
  return size_t(G) * (size_t(2) * N * N * sizeof(double2) + (NE / 2) * sizeof(Rot) + N * sizeof(double));
}

template <int N, int L>
static void launch_jacobi_n(int M, double2* A, double* W, int* info, const double* masses, hipStream_t stream) {
  constexpr int G = 64 / L;
  hipLaunchKernelGGL((k_jacobi_n<N, L>), dim3(ceil_div(M, G)), dim3(64), (jacobi_n_lds_bytes<N, L>()), stream, M, A, W,
                     info, masses, 40);
}

template <int L>
static void launch_eig_ql(int N, int M, double2* A, double* W, int* info, hipStream_t stream) {
  const size_t lds = ql_lds_bytes(N, L);
  PHX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_eig_ql<L>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              int(lds)));
  hipLaunchKernelGGL(k_eig_ql<L>, dim3(ceil_div(M, 64 / L)), dim3(64), lds, stream, N, M, A, W, info);
}

// Launch the batched eigensolver on device buffers.  Electrons (no masses):
// the tridiagonal QL kernel, with the lanes per matrix that hold its rows.
// Phonons: Jacobi, with the order fixed at compile time for 2, 4 and 6 atoms
// (6, 12 and 18 modes), packed 8 or 4 matrices per wave up to N = 12 and one per
// wave above (where 4 would hold 35 KB of LDS per workgroup and leave one wave
// per SIMD), the runtime-order kernel otherwise.
void launch_jacobi(int N, int M, double2* A, double* W, int* info, const double* masses,
                   hipStream_t stream) {
  PHX_REQUIRE(N >= 1 && N <= 64, "eigensolver supports 1 <= N <= 64");
  if (M <= 0) return;
  if (!masses) {
    if (N <= 8) launch_eig_ql<8>(N, M, A, W, info, stream);
    else if (N <= 16) launch_eig_ql<16>(N, M, A, W, info, stream);
    else if (N <= 32) launch_eig_ql<32>(N, M, A, W, info, stream);
    else launch_eig_ql<64>(N, M, A, W, info, stream);
  } else {
    switch (N) {
      case 6: launch_jacobi_n<6, 8>(M, A, W, info, masses, stream); break;
      case 12: launch_jacobi_n<12, 16>(M, A, W, info, masses, stream); break;
      case 18: launch_jacobi_n<18, 64>(M, A, W, info, masses, stream); break;
      default:
        hipLaunchKernelGGL(k_jacobi, dim3(M), dim3(64), jacobi_lds_bytes(N), stream, N, M, A, W, info, masses, 40);
    }
  }
  PHX_HIP(hipGetLastError());
}

}  // namespace phx
