// The other branches of update_factor (Cpd.hpp:189-228) on the device:
//   unconstrained   A = M V^{-1}         (Cpd.hpp:196-200; Eigen .inverse(), PartialPivLU)
//   orthogonality   A = M (M^T M)^{-1/2}  (Cpd.hpp:210-219; symmetric eigendecomposition)
// R x R work runs in one block with the matrices in LDS; every element is computed with
// the operations, in the order, of the CPU restatement (ptno_inverse, jacobi_rr,
// update_factor), so the results agree bit for bit.  Matrices are column-major R x R
// (a[i + R j]); factor rows are row-major with leading dimension ldr.
#include "ptn_internal.hpp"

namespace ptn {

namespace {

#include "wave_common.inc"

constexpr double kDblEps = 2.220446049250313e-16;

// LU with partial pivoting (the largest |entry| of the column, first one on ties), then
// the inverse column by column: pivots, forward substitution (unit lower), backward
// substitution.  A zero pivot leaves Vi as NaN.
__global__ __launch_bounds__(256) void k_lu_inverse(int R, const double *__restrict__ V, double *__restrict__ Vi) {
  __shared__ double lu[kMaxRank * kMaxRank], x[kMaxRank * kMaxRank];
  __shared__ int piv[kMaxRank];
  __shared__ int ok;
  const int t = threadIdx.x;
  for (int e = t; e < R * R; e += 256) lu[e] = V[e];
  if (t == 0) ok = 1;
  __syncthreads();
  for (int k = 0; k < R; ++k) {
    if (t == 0) {
      int p = k;
      for (int i = k + 1; i < R; ++i)
        if (fabs(lu[i + R * k]) > fabs(lu[p + R * k])) p = i;
      piv[k] = p;
      if (lu[p + R * k] == 0.0) ok = 0;
    }
    __syncthreads();
    if (!ok) break;
    const int p = piv[k];
    if (p != k)
      for (int j = t; j < R; j += 256) {
        const double tmp = lu[k + R * j];
        lu[k + R * j] = lu[p + R * j];
        lu[p + R * j] = tmp;
      }
    __syncthreads();
    for (int i = k + 1 + t; i < R; i += 256) lu[i + R * k] = lu[i + R * k] / lu[k + R * k];
    __syncthreads();
    const int m = R - k - 1;
    for (int e = t; e < m * m; e += 256) {
      const int i = k + 1 + e % m, j = k + 1 + e / m;
      lu[i + R * j] = fma(-lu[i + R * k], lu[k + R * j], lu[i + R * j]);
    }
    __syncthreads();
  }
  if (!ok) {
    for (int e = t; e < R * R; e += 256) Vi[e] = NAN;
    return;
  }
  if (t < R) {
    const int c = t;
    double *xc = x + R * c;
    for (int i = 0; i < R; ++i) xc[i] = (i == c) ? 1.0 : 0.0;
    for (int k = 0; k < R; ++k)
      if (piv[k] != k) {
        const double tmp = xc[k];
        xc[k] = xc[piv[k]];
        xc[piv[k]] = tmp;
      }
    for (int i = 0; i < R; ++i)
      for (int k = 0; k < i; ++k) xc[i] = fma(-lu[i + R * k], xc[k], xc[i]);
    for (int i = R - 1; i >= 0; --i) {
      for (int k = i + 1; k < R; ++k) xc[i] = fma(-lu[i + R * k], xc[k], xc[i]);
      xc[i] = xc[i] / lu[i + R * i];
    }
  }
  __syncthreads();
  for (int e = t; e < R * R; e += 256) Vi[e] = x[e];
}

// Parallel-order cyclic Jacobi (Golub & Van Loan 8.5, Brent-Luk round-robin order): each
// round applies the n/2 disjoint rotations, rows first (J^T A), then columns (A J) and the
// eigenvector accumulation; a rotation is skipped when |a_pq| <= eps sqrt(|a_pp a_qq|).
// Up to 60 sweeps, stopping after a sweep without rotations.  evals = diag, Q = vectors.
//
// The chain of rounds bounds it (n - 1 rounds a sweep, some 8 sweeps), and a round is two halves
// of some 1000 clocks.  In the first the lanes of a wave of their own form the rotations side by
// side (divisions and square roots, the short ones where the operands allow); meanwhile the
// other four waves fetch the round's entries, a 2 x 2 block to a thread, the rows of one pair by the
// columns of another, and apply the round before to the vectors.  In the second they apply both
// rotations to their blocks in registers, rows first, with no barrier between the two and no
// branch on which pairs rotate.  A pair's members move on by one slot a round (the first stays), so
// no round computes them.  R = 24: 1161 us with one thread's rotations and six barriers a round,
// 199 with the rotations side by side before the blocks and the vectors, 163 so.  RB: R rounded up
// to 16, 32 or 64, so that a thread's blocks are fixed before the loop.
template <int RB>
__global__ __launch_bounds__(320) void k_jacobi_eig(int R, const double *__restrict__ A, double *__restrict__ evals,
                                                    double *__restrict__ Q) {
  __shared__ double a[RB * RB], v[RB * RB];
  __shared__ double cs[2][RB / 2], sn[2][RB / 2];   // of this round and the last
  __shared__ unsigned long long act;                 // the pairs that rotate this round
  constexpr int NA = (RB / 2 * (RB / 2) + 255) / 256, NV = (RB * (RB / 2) + 255) / 256;
  const int t = threadIdx.x;
  const int n = R + (R & 1), U = n / 2;              // odd R: the pair with index R stands still
  // pair k of round r: slots k and n - 1 - k, where slot 0 holds 0 and the others turn
  struct Pair {
    int k, x, y;
    __device__ int p() const { return x < y ? x : y; }
    __device__ int q() const { return x < y ? y : x; }
  };
  auto pair = [&](int k) { return Pair{k, k, n - 1 - k}; };
  auto turn = [&](Pair &P) {
    P.x = P.k == 0 ? 0 : P.x == n - 1 ? 1 : P.x + 1;
    P.y = P.y == n - 1 ? 1 : P.y + 1;
  };
  for (int e = t; e < R * R; e += 320) {
    a[e] = A[e];
    v[e] = (e % R == e / R) ? 1.0 : 0.0;
  }
  if (t >= 256) {                                    // the rotations
    const int l = t - 256;
    Pair P = pair(l < U ? l : 0);
    int par = 0;
    for (int sweep = 0; sweep < 60; ++sweep) {
      bool rotated = false;
      for (int r = 0; r < n - 1; ++r) {
        const int p = P.p(), q = P.q();
        const bool whole = l < U && q < R;
        const int qc = q < R ? q : p;
        __syncthreads();                             // the last round's blocks are stored
        const double apq = a[p + R * qc], app = a[p + R * p], aqq = a[qc + R * qc];
        // lanes without a rotation take the numbers of one, so that the wave need not leave the
        // short operations for them
        const bool some = whole && apq != 0.0;
        const double den = some ? 2.0 * apq : 2.0, num = some ? aqq - app : 0.0, pr = some ? fabs(app * aqq) : 1.0;
        double small, cc, ss;
        bool plain = !(mid_range(den) && mid_range(pr) && (num == 0.0 || mid_range(num)));
        const double th = short_quotient(num, den);
        plain |= !(fabs(th) < 0x1p199);
        if (!__any(plain)) {
          small = kDblEps * short_sqrt(pr);
          double tt = short_quotient(1.0, fabs(th) + short_sqrt(fma(th, th, 1.0)));
          tt = th < 0.0 ? -tt : tt;
          cc = short_quotient(1.0, short_sqrt(fma(tt, tt, 1.0)));
          ss = tt * cc;
        } else {
          small = kDblEps * sqrt(pr);
          const double theta = num / den;
          double tt = 1.0 / (fabs(theta) + sqrt(fma(theta, theta, 1.0)));
          if (fabs(theta) > 1e150) tt = 0.5 / theta;
          else if (theta < 0.0) tt = -tt;
          cc = 1.0 / sqrt(fma(tt, tt, 1.0));
          ss = tt * cc;
        }
        const bool on = whole && !(apq == 0.0 || fabs(apq) <= small);
        if (on) {
          cs[par][l] = cc;
          sn[par][l] = ss;
        }
        const unsigned long long m = __ballot(on);
        if (l == 0) act = m;
        __syncthreads();
        rotated |= m != 0;
        turn(P);
        par ^= 1;
      }
      if (!rotated) break;                           // the same in every wave
    }
  } else {
    Pair ra[NA], ca[NA], cv[NV];                     // blocks (row pair, column pair); (row of v, pair)
    int vi[NV];
#pragma unroll
    for (int u = 0; u < NA; ++u) {
      const int e = t + 256 * u;
      ra[u] = pair(e < U * U ? e % U : 0);
      ca[u] = pair(e < U * U ? e / U : 0);
    }
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int e = t + 256 * u;
      vi[u] = e < R * U ? e % R : -1;
      cv[u] = pair(e < R * U ? e / R : 0);
    }
    // the rotations of round `par`, pairs m, applied to the vectors
    auto vectors = [&](unsigned long long m, int par) {
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        const int k = cv[u].k;
        if (vi[u] >= 0 && ((m >> k) & 1)) {
          const int i = vi[u], p = cv[u].p(), q = cv[u].q();
          const double c = cs[par][k], s = sn[par][k], vx = v[i + R * p], vy = v[i + R * q];
          v[i + R * p] = fma(c, vx, -(s * vy));
          v[i + R * q] = fma(s, vx, c * vy);
        }
        turn(cv[u]);
      }
    };
    unsigned long long last = 0;                     // the pairs of the round before
    int par = 0;
    bool first = true;
    for (int sweep = 0; sweep < 60; ++sweep) {
      bool rotated = false;
      for (int r = 0; r < n - 1; ++r) {
        double x00[NA], x10[NA], x01[NA], x11[NA];
        int e00[NA], e10[NA], e01[NA], e11[NA];
        bool hq[NA], hq2[NA];                        // (a standing pair has one member: its other reads it too)
        __syncthreads();                             // the last round's blocks are stored
#pragma unroll
        for (int u = 0; u < NA; ++u) {
          const int p = ra[u].p(), p2 = ca[u].p();
          hq[u] = ra[u].q() < R;
          hq2[u] = ca[u].q() < R;
          const int q = hq[u] ? ra[u].q() : p, q2 = hq2[u] ? ca[u].q() : p2;
          e00[u] = p + R * p2;
          e10[u] = q + R * p2;
          e01[u] = p + R * q2;
          e11[u] = q + R * q2;
          x00[u] = a[e00[u]];
          x10[u] = a[e10[u]];
          x01[u] = a[e01[u]];
          x11[u] = a[e11[u]];
          turn(ra[u]);
          turn(ca[u]);
        }
        if (!first) vectors(last, par ^ 1);
        first = false;
        __syncthreads();
        const unsigned long long m = act;
        double cr[NA], sr[NA], cc[NA], sc[NA];
#pragma unroll
        for (int u = 0; u < NA; ++u) {
          cr[u] = cs[par][ra[u].k];
          sr[u] = sn[par][ra[u].k];
          cc[u] = cs[par][ca[u].k];
          sc[u] = sn[par][ca[u].k];
        }
        if (m != 0) {
          rotated = true;
#pragma unroll
          for (int u = 0; u < NA; ++u) {
            if (t + 256 * u >= U * U) continue;
            const int kr = ra[u].k, kc = ca[u].k;
            const bool ron = (m >> kr) & 1, con = (m >> kc) & 1;
            {                                        // rows p, q (a pair that rotates has both)
              const double c = cr[u], s = sr[u];
              const double y00 = fma(c, x00[u], -(s * x10[u])), y10 = fma(s, x00[u], c * x10[u]);
              const double y01 = fma(c, x01[u], -(s * x11[u])), y11 = fma(s, x01[u], c * x11[u]);
              x00[u] = ron ? y00 : x00[u];
              x10[u] = ron ? y10 : x10[u];
              x01[u] = ron ? y01 : x01[u];
              x11[u] = ron ? y11 : x11[u];
            }
            {                                        // columns p2, q2
              const double c = cc[u], s = sc[u];
              const double y00 = fma(c, x00[u], -(s * x01[u])), y01 = fma(s, x00[u], c * x01[u]);
              const double y10 = fma(c, x10[u], -(s * x11[u])), y11 = fma(s, x10[u], c * x11[u]);
              const bool own = con && kr == kc;      // the rotated pair's own entries: zero
              x00[u] = con ? y00 : x00[u];
              x10[u] = own ? 0.0 : con ? y10 : x10[u];
              x01[u] = own ? 0.0 : con ? y01 : x01[u];
              x11[u] = con ? y11 : x11[u];
            }
            a[e00[u]] = x00[u];
            if (hq[u]) a[e10[u]] = x10[u];
            if (hq2[u]) a[e01[u]] = x01[u];
            if (hq[u] && hq2[u]) a[e11[u]] = x11[u];
          }
        }
        last = m;
        par ^= 1;
      }
      if (!rotated) break;
    }
    vectors(last, par ^ 1);
  }
  __syncthreads();
  for (int e = t; e < R * R; e += 320) Q[e] = v[e];
  for (int i = t; i < R; i += 320) evals[i] = a[i + R * i];
}

// T[a][b] = sum_k Q[a][k] sqrt(1 / ev[k]) Q[b][k]  ((M^T M)^{-1/2})
__global__ void k_inv_sqrt(int R, const double *__restrict__ Q, const double *__restrict__ ev, double *__restrict__ T) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= R * R) return;
  const int a = e % R, b = e / R;
  double s = 0.0;
  for (int k = 0; k < R; ++k) s = fma(Q[a + R * k] * sqrt(1.0 / ev[k]), Q[b + R * k], s);
  T[a + R * b] = s;
}

// A[i][c] = sum_k M[i][k] T[k][c] (rows of ldr doubles, columns beyond R left as they are)
__global__ void k_apply_right(int64_t I, int R, int ldr, const double *__restrict__ M, const double *__restrict__ T,
                              double *__restrict__ A) {
  const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (e >= I * R) return;
  const int64_t i = e / R;
  const int c = (int)(e - i * R);
  double s = 0.0;
  for (int k = 0; k < R; ++k) s = fma(M[i * ldr + k], T[k + R * c], s);
  A[i * ldr + c] = s;
}

// the Nesterov log fields of a mode updated without NNLS
__global__ void k_params_no_nnls(NnlsParams *p) {
  if (threadIdx.x == 0) {
    p->L0 = 0.0;
    p->mu0 = 0.0;
    p->iters = 0;
    p->fallback = 0;
    p->warm_rows = 0;
    p->warm_steps = 0;
  }
}

}  // namespace

void lu_inverse(hipStream_t s, int R, const double *V, double *Vi) { k_lu_inverse<<<1, 256, 0, s>>>(R, V, Vi); }

void jacobi_eig(hipStream_t s, int R, const double *A, double *evals, double *Q) {
  if (R <= 16) k_jacobi_eig<16><<<1, 320, 0, s>>>(R, A, evals, Q);
  else if (R <= 32) k_jacobi_eig<32><<<1, 320, 0, s>>>(R, A, evals, Q);
  else k_jacobi_eig<64><<<1, 320, 0, s>>>(R, A, evals, Q);
}

void inv_sqrt_matrix(hipStream_t s, int R, const double *Q, const double *ev, double *T) {
  k_inv_sqrt<<<(R * R + 255) / 256, 256, 0, s>>>(R, Q, ev, T);
}

void apply_right(hipStream_t s, int64_t I, int R, int ldr, const double *M, const double *T, double *A) {
  k_apply_right<<<(unsigned)((I * R + 255) / 256), 256, 0, s>>>(I, R, ldr, M, T, A);
}

void params_no_nnls(hipStream_t s, NnlsParams *p) { k_params_no_nnls<<<1, 64, 0, s>>>(p); }

}  // namespace ptn
