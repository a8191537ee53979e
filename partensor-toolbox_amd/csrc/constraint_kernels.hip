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

__device__ __forceinline__ int rr_slot(int k, int t, int n) { return k == 0 ? 0 : ((k - 1 + t) % (n - 1)) + 1; }

// Parallel-order cyclic Jacobi (Golub & Van Loan 8.5, Brent-Luk round-robin order): each
// round applies the n/2 disjoint rotations, rows first (J^T A), then columns (A J) and the
// eigenvector accumulation; a rotation is skipped when |a_pq| <= eps sqrt(|a_pp a_qq|).
// Up to 60 sweeps, stopping after a sweep without rotations.  evals = diag, Q = vectors.
//
// The chain of rounds bounds it (n - 1 rounds a sweep, some 8 sweeps), so a round is made
// short: lane k of the first wave forms rotation k (its divisions and square roots side by
// side with the others' instead of one after another on one thread), and a thread applies a
// round to one 2 x 2 block at a time, the rows of one pair by the columns of another, in
// registers: rows first, then columns, as before, with no barrier between the two.  Two
// barriers a round instead of six; R = 24: 1161 -> 199 us.  RB: R rounded up to 16, 32 or 64,
// so that a thread's blocks are fixed before the loop.
template <int RB>
__global__ __launch_bounds__(256) void k_jacobi_eig(int R, const double *__restrict__ A, double *__restrict__ evals,
                                                    double *__restrict__ Q) {
  __shared__ double a[RB * RB], v[RB * RB];
  __shared__ double cs[RB / 2], sn[RB / 2];
  __shared__ int pp[RB / 2], qq[RB / 2];
  __shared__ unsigned long long act;                 // the pairs that rotate this round
  constexpr int NA = (RB / 2 * (RB / 2) + 255) / 256, NV = (RB * (RB / 2) + 255) / 256;
  const int t = threadIdx.x;
  const int n = R + (R & 1), U = n / 2;              // odd R: the pair with index R stands still
  int ma[NA], mb[NA], vi[NV], vm[NV];                // blocks (row pair, column pair) and (row of v, pair)
#pragma unroll
  for (int u = 0; u < NA; ++u) {
    const int e = t + 256 * u;
    ma[u] = e < U * U ? e % U : -1;
    mb[u] = e / U;
  }
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int e = t + 256 * u;
    vi[u] = e < R * U ? e % R : -1;
    vm[u] = e / R;
  }
  for (int e = t; e < R * R; e += 256) {
    a[e] = A[e];
    v[e] = (e % R == e / R) ? 1.0 : 0.0;
  }
  for (int sweep = 0; sweep < 60; ++sweep) {
    bool rotated = false;
    for (int r = 0; r < n - 1; ++r) {
      __syncthreads();                               // the last round's blocks are stored
      if (t < 64) {
        int p = 0, q = 0;
        bool on = t < U;
        double cc = 1.0, ss = 0.0;
        if (on) {
          p = rr_slot(t, r, n);
          q = rr_slot(n - 1 - t, r, n);
          if (p > q) {
            const int tmp = p;
            p = q;
            q = tmp;
          }
          pp[t] = p;
          qq[t] = q;
          on = q < R;
        }
        if (on) {
          const double apq = a[p + R * q], app = a[p + R * p], aqq = a[q + R * q];
          if (apq == 0.0 || fabs(apq) <= kDblEps * sqrt(fabs(app * aqq))) {
            on = false;
          } else {
            const double theta = (aqq - app) / (2.0 * apq);
            double tt;
            if (fabs(theta) > 1e150) tt = 0.5 / theta;
            else {
              tt = 1.0 / (fabs(theta) + sqrt(fma(theta, theta, 1.0)));
              if (theta < 0.0) tt = -tt;
            }
            cc = 1.0 / sqrt(fma(tt, tt, 1.0));
            ss = tt * cc;
            cs[t] = cc;
            sn[t] = ss;
          }
        }
        const unsigned long long m = __ballot(on);
        if (t == 0) act = m;
      }
      __syncthreads();
      const unsigned long long m = act;
      if (m == 0) continue;                          // uniform: written again after the next barrier
      rotated = true;
#pragma unroll
      for (int u = 0; u < NA; ++u) {
        if (ma[u] < 0) continue;
        const bool ron = (m >> ma[u]) & 1, con = (m >> mb[u]) & 1;
        if (!ron && !con) continue;
        const int p = pp[ma[u]], q = qq[ma[u]], p2 = pp[mb[u]], q2 = qq[mb[u]];
        const bool hq = q < R, hq2 = q2 < R;         // (a standing pair has one member)
        double x00 = a[p + R * p2], x10 = hq ? a[q + R * p2] : 0.0;
        double x01 = hq2 ? a[p + R * q2] : 0.0, x11 = hq && hq2 ? a[q + R * q2] : 0.0;
        if (ron) {                                   // rows p, q
          const double c = cs[ma[u]], s = sn[ma[u]];
          const double y00 = fma(c, x00, -(s * x10)), y10 = fma(s, x00, c * x10);
          const double y01 = fma(c, x01, -(s * x11)), y11 = fma(s, x01, c * x11);
          x00 = y00;
          x10 = y10;
          x01 = y01;
          x11 = y11;
        }
        if (con) {                                   // columns p2, q2
          const double c = cs[mb[u]], s = sn[mb[u]];
          const double y00 = fma(c, x00, -(s * x01)), y01 = fma(s, x00, c * x01);
          const double y10 = fma(c, x10, -(s * x11)), y11 = fma(s, x10, c * x11);
          x00 = y00;
          x10 = y10;
          x01 = y01;
          x11 = y11;
          if (ma[u] == mb[u]) x01 = x10 = 0.0;
        }
        a[p + R * p2] = x00;
        if (hq) a[q + R * p2] = x10;
        if (hq2) a[p + R * q2] = x01;
        if (hq && hq2) a[q + R * q2] = x11;
      }
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        if (vi[u] < 0 || !((m >> vm[u]) & 1)) continue;
        const int i = vi[u], p = pp[vm[u]], q = qq[vm[u]];
        const double c = cs[vm[u]], s = sn[vm[u]];
        const double vx = v[i + R * p], vy = v[i + R * q];
        v[i + R * p] = fma(c, vx, -(s * vy));
        v[i + R * q] = fma(s, vx, c * vy);
      }
    }
    if (!rotated) break;                             // uniform
  }
  __syncthreads();
  for (int e = t; e < R * R; e += 256) Q[e] = v[e];
  for (int i = t; i < R; i += 256) evals[i] = a[i + R * i];
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
  if (R <= 16) k_jacobi_eig<16><<<1, 256, 0, s>>>(R, A, evals, Q);
  else if (R <= 32) k_jacobi_eig<32><<<1, 256, 0, s>>>(R, A, evals, Q);
  else k_jacobi_eig<64><<<1, 256, 0, s>>>(R, A, evals, Q);
}

void inv_sqrt_matrix(hipStream_t s, int R, const double *Q, const double *ev, double *T) {
  k_inv_sqrt<<<(R * R + 255) / 256, 256, 0, s>>>(R, Q, ev, T);
}

void apply_right(hipStream_t s, int64_t I, int R, int ldr, const double *M, const double *T, double *A) {
  k_apply_right<<<(unsigned)((I * R + 255) / 256), 256, 0, s>>>(I, R, ldr, M, T, A);
}

void params_no_nnls(hipStream_t s, NnlsParams *p) { k_params_no_nnls<<<1, 64, 0, s>>>(p); }

}  // namespace ptn
