// R x R and row-wise pieces of an ALS update, all FP64 on the device:
// Gram Hadamard products (PartialCwiseProd.hpp:54-222), Grams (Cpd.hpp:227),
// extreme singular values of V + GLambda (NesterovMNLS.hpp:45-91), the batched
// Nesterov NNLS (NesterovMNLS.hpp:181-234), the zero-column blend
// (Cpd.hpp:206-207), Normalize (Normalize.hpp:92-174), the Gram-form costs
// (CpdCUDA.hpp:137-142, Cpd.hpp:162-169) and the acceleration extrapolation
// (Cpd.hpp:247-258).  Built with -ffp-contract=off: fused multiply-adds appear
// only where written as fma(), so the arithmetic sequence is fixed.
#include "ptn_internal.hpp"

namespace ptn {

namespace {

typedef double f64x2 __attribute__((ext_vector_type(2)));

struct GramPtrs {
  const double *p[kMaxOrder];
};
#include "wave_common.inc"

struct MutPtrs {
  double *p[kMaxOrder];
};

// Accumulate in list order: V = G_l0; V = G_lj * V (right-nested when the list is
// ascending, left-nested along a tree path when given in path order).
__global__ void k_hadamard(int R, int ng, GramPtrs G, double *V) {
  for (int e = threadIdx.x; e < R * R; e += blockDim.x) {
    double v = G.p[0][e];
    for (int j = 1; j < ng; ++j) v = G.p[j][e] * v;
    V[e] = v;
  }
}

// G = A^T A: block c sums rows [32c, 32c+32) in order for every entry (4 x 4 entries
// per thread, rows staged in LDS, missing rows padded with zeros, which add exact
// zeros); k_gram_combine adds the chunk sums in order.  Same association as the CPU
// restatement.
__device__ __forceinline__ void gram_rows32(const double (*As)[kMaxRank + 4], int R, int tid, double *o) {
  const int nb = (R + 3) / 4;                 // 4-wide blocks per dimension
  if (tid >= nb * nb) return;
  const int a0 = 4 * (tid / nb), b0 = 4 * (tid % nb);
  double acc[4][4];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) acc[x][y] = 0.0;
#pragma unroll 8
  for (int i = 0; i < 32; ++i) {
    double va[4], vb[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) { va[x] = As[i][a0 + x]; vb[x] = As[i][b0 + x]; }
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int y = 0; y < 4; ++y) acc[x][y] = fma(va[x], vb[y], acc[x][y]);
  }
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y)
      if (a0 + x < R && b0 + y < R) o[(a0 + x) * R + b0 + y] = acc[x][y];
}

// Rows [i0, i0 + 32) of a factor (ldr = 16 NT doubles a row, consecutive) into As, zeros past I
// and past R: each thread's NT 16-byte loads are in flight together.  The kernels that use it
// (a few blocks, a few rows each) are bound by such latencies: one element at a time through
// an index division they waited for each load (800 rows, R = 32 beside the tensor passes:
// k_gram_chunks 22 -> 12 us, k_nnls_finish 22 -> 14; 100 rows, R = 10: 6.3 -> 4.3, 8.3 -> 5.2).
template <int NT>
__device__ __forceinline__ void load_rows32(const double *__restrict__ A, int64_t i0, int64_t I, int R,
                                            double (*As)[kMaxRank + 4], double *__restrict__ copy) {
  constexpr int LDR = 16 * NT, H = LDR / 2;
  f64x2 v[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    const int e = threadIdx.x + 256 * u, i = e / H, c = 2 * (e % H);
    v[u] = f64x2{0.0, 0.0};
    if (i0 + i < I) v[u] = *(const f64x2 *)(A + (i0 + i) * LDR + c);
  }
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    const int e = threadIdx.x + 256 * u, i = e / H, c = 2 * (e % H);
    if (copy && i0 + i < I) *(f64x2 *)(copy + (i0 + i) * LDR + c) = v[u];
    As[i][c] = c < R ? v[u][0] : 0.0;
    As[i][c + 1] = c + 1 < R ? v[u][1] : 0.0;
  }
}

template <int NT>
__global__ __launch_bounds__(256) void k_gram_chunks(int64_t I, int R, const double *__restrict__ A,
                                                     double *__restrict__ partials) {
  __shared__ __align__(16) double As[32][kMaxRank + 4];
  load_rows32<NT>(A, (int64_t)blockIdx.x * 32, I, R, As, nullptr);
  __syncthreads();
  gram_rows32(As, R, threadIdx.x, partials + (int64_t)blockIdx.x * R * R);
}

// the sum of entry e over the chunk partials, in order, eight loads in flight
__device__ __forceinline__ double combine_chunks(const double *__restrict__ partials, int e, int RR, int nchunks) {
  double g = partials[e];
  int c = 1;
  for (; c + 8 <= nchunks; c += 8) {
    double p[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) p[j] = partials[(int64_t)(c + j) * RR + e];
#pragma unroll
    for (int j = 0; j < 8; ++j) g = g + p[j];
  }
  for (; c < nchunks; ++c) g = g + partials[(int64_t)c * RR + e];
  return g;
}

__global__ __launch_bounds__(256) void k_gram_combine(int R, int nchunks, const double *__restrict__ partials,
                                                      double *__restrict__ G) {
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < R * R; e += gridDim.x * blockDim.x)
    G[e] = combine_chunks(partials, e, R * R, nchunks);
}

// The Grams of all factors and the Hadamard product of some of them (the line search's: A_hat's
// Grams and V_hat) in two launches: block b sums one 32-row chunk of one factor, then wave k
// of a block combines 64 entries of factor k's Gram in k_gram_combine's order and the first
// wave multiplies the ng listed ones in list order (k_hadamard's).  Two launches per factor
// and one for the product kept the line search of small tensors waiting for the side stream
// (100^3, R = 10, 50 sweeps 14.7 -> 13.8 ms).
struct GramBatch {
  int N, ng;
  int64_t I[kMaxOrder];
  int chunk0[kMaxOrder + 1];                   // first chunk of each factor, then their number
  const double *A[kMaxOrder];
  double *G[kMaxOrder];
  int list[kMaxOrder];
};
template <int NT>
__global__ __launch_bounds__(256) void k_gram_chunks_all(GramBatch b, int R, double *__restrict__ partials) {
  __shared__ __align__(16) double As[32][kMaxRank + 4];
  int k = 0;
  while (k + 1 < b.N && (int)blockIdx.x >= b.chunk0[k + 1]) ++k;
  load_rows32<NT>(b.A[k], (int64_t)((int)blockIdx.x - b.chunk0[k]) * 32, b.I[k], R, As, nullptr);
  __syncthreads();
  gram_rows32(As, R, threadIdx.x, partials + (int64_t)blockIdx.x * R * R);
}
__global__ __launch_bounds__(64 * kMaxOrder) void k_gram_combine_all(GramBatch b, int R,
                                                                     const double *__restrict__ partials,
                                                                     double *__restrict__ V) {
  __shared__ double g[kMaxOrder][64];
  const int lane = threadIdx.x & 63, k = threadIdx.x >> 6, e = blockIdx.x * 64 + lane;
  if (e < R * R) {
    const double v = combine_chunks(partials + (int64_t)b.chunk0[k] * R * R, e, R * R, b.chunk0[k + 1] - b.chunk0[k]);
    b.G[k][e] = v;
    g[k][lane] = v;
  }
  __syncthreads();
  if (k == 0 && e < R * R) {
    double v = g[b.list[0]][lane];
    for (int j = 1; j < b.ng; ++j) v = g[b.list[j]][lane] * v;
    V[e] = v;
  }
}

// With ng > 0 the matrix is first formed as the Hadamard product of the ng Grams in
// list order (V = G_l0, V = G_lj * V; PartialCwiseProd) and stored to Vout; with
// betas != nullptr the momentum coefficients of the Nesterov solve follow the
// eigenvalues (one kernel prepares an NNLS update).  One block.
template <int RB>
__global__ __launch_bounds__(kEigThreads<RB>) void k_eig_extremes(int R, const double *__restrict__ V, GramPtrs G, int ng,
                                                      double *__restrict__ Vout, NnlsParams *prm, int max_inner,
                                                      double *__restrict__ betas) {
  __shared__ EigLds<RB> S;
  const int n = R;
  for (int x = threadIdx.x; x < RB * RB; x += kEigThreads<RB>) {
    const int r = x / RB, c = x % RB;
    double v = 0.0;
    if (r < n && c < n) {
      const int e = r * n + c;
      if (ng > 0) {
        v = G.p[0][e];
        for (int j = 1; j < ng; ++j) v = G.p[j][e] * v;
        Vout[e] = v;
      } else {
        v = V[e];
      }
    }
    S.t[x] = v;
  }
  __syncthreads();
  double amax, amin;
  eig_extremes_block<RB>(n, S, amax, amin);
  if (threadIdx.x < 64) glambda_betas(amax, amin, prm, max_inner, betas);
}



// One 64-lane wave per factor row; lane r (mod RB) holds column r and keeps column r of
// Zt = V + lambda I in registers.  Each step the row y is broadcast through LDS and
// (Y Zt)(i, r) accumulates four interleaved partial sums over k mod 4, combined
// pairwise, as the CPU restatement does; lanes and k beyond R hold exact zeros, which
// leave the sums unchanged.  Each lane records whether its entry passes the stop test
// (NesterovMNLS.hpp:217) at every check; the row's mask is the AND over its lanes
// (max |G.Y| <= d1 and min G >= -d2 hold iff they hold entry-wise).  Iterate A_k goes
// to hist[k]; the common stopping point is selected afterwards.  The momentum
// coefficients depend only on q and come precomputed (momentum_wave).
//
// The chain of steps bounds it, and a step is as long as what a wave issues in it.  With R <= 32 the
// 64 lanes hold two or four copies of the row, and each copy forms its own two or one of the
// four partial sums (all four by every copy: 100 rows at rank 10 15.0 us, so 12.5; 301 at 24 21.0
// and 16.3).
template <int RB>
__global__ __launch_bounds__(256) void k_nnls_iterate(int64_t I, int R, int ldr, const double *__restrict__ V,
                                                      const NnlsParams *__restrict__ prm,
                                                      const double *__restrict__ betas,
                                                      const double *__restrict__ M, const double *__restrict__ A,
                                                      const double *__restrict__ S, double d1, double d2, int max_inner,
                                                      unsigned long long *mask, double *__restrict__ hist,
                                                      double *colsum) {
  __shared__ double sbeta[kMaxInner + 1];
  if (blockIdx.x == 0 && (int)threadIdx.x < R) colsum[threadIdx.x] = 0.0;   // summed by k_nnls_select
  constexpr int GP = 64 / RB, NC = 4 / GP, NR = RB / 4;   // groups of RB lanes; chains of a group, their length
  // y, by chain where a group has some of them: y_k at SQ (k mod 4) + SJ (k / 4)
  constexpr int SQ = RB == 64 ? 1 : NR, SJ = RB == 64 ? 4 : 1;
  __shared__ __align__(16) double ybuf[4][RB];
  __shared__ unsigned long long wbits[4][4];
  for (int k = threadIdx.x; k < max_inner; k += blockDim.x) sbeta[k] = betas[k];
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave;
  unsigned long long bits[4] = {~0ull, ~0ull, ~0ull, ~0ull};
  if (row < I) {
  const double lambda = prm->lambda, L = prm->L;
  const double invL = 1.0 / L;
  const int c = lane % RB, grp = RB == 64 ? 0 : lane / RB;
  const bool on = c < R;
  const int r = on ? c : 0;
  double z[NC][NR];
#pragma unroll
  for (int q = 0; q < NC; ++q)
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      const int k = 4 * j + grp * NC + q;
      const double vk = (on && k < R) ? V[k * R + r] : 0.0;
      z[q][j] = (k == r && on) ? vk + lambda : vk;
    }
  // lanes >= R: zero start, zero column of Zt and zero Wt keep every iterate at +0.
  // The anchor of W~ is always the previous row A; the start is A or the warm start S.
  const double anc = on ? A[row * ldr + r] : 0.0;
  const double a0 = on ? (S ? S[row * ldr + r] : anc) : 0.0;
  const double wt = on ? M[row * ldr + r] + lambda * anc : 0.0;
  double y = a0, acur = a0;
  const int64_t hstride = I * ldr;
  double *hrow = hist + row * ldr + lane;
  if (lane < ldr) hrow[0] = a0;
  for (int kw = 0; kw < 4; ++kw) {
    unsigned long long m = 0ull;
    const int kend = max_inner - 64 * kw < 64 ? max_inner - 64 * kw : 64;
    for (int kb = 0; kb < kend; ++kb) {
      const int k = 64 * kw + kb;
      const double beta = sbeta[k];
      if (lane < RB) ybuf[wave][SQ * (c & 3) + SJ * (c >> 2)] = y;
      __builtin_amdgcn_wave_barrier();
      double sq[NC];
#pragma unroll
      for (int q = 0; q < NC; ++q) sq[q] = 0.0;
      const double *yb = ybuf[wave] + (RB == 64 ? 0 : grp * NC * NR);
#pragma unroll
      for (int j = 0; j < NR; ++j)
#pragma unroll
        for (int q = 0; q < NC; ++q) sq[q] = fma(yb[SQ * q + SJ * j], z[q][j], sq[q]);
      __builtin_amdgcn_wave_barrier();
      double dot;
      if constexpr (RB == 16) dot = add_other_half<32>(add_other_half<16>(sq[0]));
      else if constexpr (RB == 32) dot = add_other_half<32>(sq[0] + sq[1]);
      else dot = (sq[0] + sq[1]) + (sq[2] + sq[3]);
      const double g = dot - wt;
      const bool fail = on && ((fabs(g * y) > d1) || (g < -d2));
      if (__ballot(fail) == 0ull) m |= 1ull << kb;       // the row passes check k
      // g / L as RN(g / L): reciprocal, then one exact-residual correction (Markstein)
      const double q0 = g * invL;
      const double tq = y - fma(fma(-q0, L, g), invL, q0);
      const double an = tq > 0.0 ? tq : 0.0;
      y = (1.0 + beta) * an - beta * acur;
      acur = an;
      if (lane < ldr) hrow[(k + 1) * hstride] = acur;
    }
    bits[kw] = m;
  }
  }
  // the block's mask (AND over its rows) goes to its own slot: no atomics
  if (lane == 0)
    for (int w = 0; w < 4; ++w) wbits[wave][w] = bits[w];
  __syncthreads();
  if (threadIdx.x < 4) {
    const int w = threadIdx.x;
    unsigned long long m = ((wbits[0][w] & wbits[1][w]) & wbits[2][w]) & wbits[3][w];
    const int lo = w * 64;
    if (max_inner < lo + 64) m |= (max_inner <= lo) ? ~0ull : (~0ull << (max_inner - lo));
    mask[(int64_t)blockIdx.x * 4 + w] = m;
  }
}

__device__ __forceinline__ int first_common_check(const unsigned long long *mask, int max_inner) {
  for (int w = 0; w < 4; ++w) {
    unsigned long long m = mask[w];
    if (m) {
      int k = w * 64 + __builtin_ctzll(m);
      return k < max_inner ? k : max_inner;
    }
  }
  return max_inner;
}

// A_new = the iterate at the first check every row satisfies (else after max_inner
// steps); column abs-sums for the zero-column test (an exact-zero test, so the
// summation order does not matter).
__global__ __launch_bounds__(256) void k_nnls_select(int64_t I, int R, int ldr, const double *__restrict__ hist,
                                                     const unsigned long long *__restrict__ mask, int max_inner,
                                                     double *__restrict__ Anew, double *colsum, NnlsParams *prm) {
  __shared__ double red[4][kMaxRank];
  __shared__ unsigned long long mred[256];
  __shared__ int sk;
  {
    // AND of the per-block masks of k_nnls_iterate (4 words per block)
    const int64_t nblk = (I + 3) / 4;
    unsigned long long m = ~0ull;
    for (int64_t b = threadIdx.x >> 2; b < nblk; b += 64) m &= mask[b * 4 + (threadIdx.x & 3)];
    mred[threadIdx.x] = m;
    __syncthreads();
    for (int o = 128; o >= 4; o >>= 1) {
      if ((int)threadIdx.x < o) mred[threadIdx.x] &= mred[threadIdx.x + o];
      __syncthreads();
    }
    if (threadIdx.x == 0) sk = first_common_check(mred, max_inner);
    __syncthreads();
  }
  const int kstar = sk;
  if (blockIdx.x == 0 && threadIdx.x == 0) prm->iters = kstar;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const double *src = hist + (int64_t)kstar * I * ldr;
  double cs = 0.0;
  for (int64_t row = (int64_t)blockIdx.x * 4 + wave; row < I; row += (int64_t)gridDim.x * 4) {
    if (lane < ldr) {
      const double v = src[row * ldr + lane];
      Anew[row * ldr + lane] = v;
      cs += fabs(v);
    }
  }
  red[wave][lane] = cs;
  __syncthreads();
  if (wave == 0 && lane < R) atomicAdd(&colsum[lane], ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane]);
}

// the zero-column fallback's mix (Cpd.hpp:206-207)
__device__ __forceinline__ double zero_col_mix(double a, double aold) { return 0.9 * a + 0.1 * aold; }

// k_nnls_select over the rows [32 b, 32 b + 32) of block b, which also leaves the
// block's partial Gram of the selected rows (k_gram_chunks' association) in
// partials[b]; k_gram_finish applies the zero-column test and combines.
template <int NT>
__global__ __launch_bounds__(256) void k_nnls_finish(int64_t I, int R, const double *__restrict__ hist,
                                                     const unsigned long long *__restrict__ mask, int max_inner,
                                                     double *__restrict__ Anew, double *colsum,
                                                     double *__restrict__ partials, NnlsParams *prm) {
  constexpr int LDR = 16 * NT;
  __shared__ __align__(16) double As[32][kMaxRank + 4];
  __shared__ unsigned long long wmask[4][4];
  const int tid = threadIdx.x;
  {
    // the AND of the blocks' masks, four words each: lane l takes word l % 4 of every 64th
    // block, the lanes of a wave meet in shuffles, the waves in LDS (one barrier)
    const int64_t nblk = (I + 3) / 4;
    unsigned long long m = ~0ull;
    for (int64_t b = tid >> 2; b < nblk; b += 64) m &= mask[b * 4 + (tid & 3)];
#pragma unroll
    for (int o = 4; o < 64; o <<= 1) m &= __shfl_xor(m, o, 64);
    if ((tid & 63) < 4) wmask[tid >> 6][tid & 3] = m;
    __syncthreads();
  }
  unsigned long long all[4];
#pragma unroll
  for (int w = 0; w < 4; ++w) all[w] = ((wmask[0][w] & wmask[1][w]) & wmask[2][w]) & wmask[3][w];
  const int kstar = first_common_check(all, max_inner);
  if (blockIdx.x == 0 && tid == 0) prm->iters = kstar;
  load_rows32<NT>(hist + (int64_t)kstar * I * LDR, (int64_t)blockIdx.x * 32, I, R, As, Anew);
  __syncthreads();
  if (tid < R) {
    double cs = 0.0;
#pragma unroll 8
    for (int i = 0; i < 32; ++i) cs += fabs(As[i][tid]);
    atomicAdd(&colsum[tid], cs);
  }
  gram_rows32(As, R, tid, partials + (int64_t)blockIdx.x * R * R);
}

// G = A^T A from the chunk partials (k_gram_combine's order), after the zero-column test
// of update_factor (Cpd.hpp:206-207): when some column abs-sum is zero, block 0 alone
// recomputes G from the mixed rows 0.9 A + 0.1 A_old in the same association and then
// stores the mixed rows.  prm->fallback records the test.
__global__ __launch_bounds__(256) void k_gram_finish(int64_t I, int R, int ldr, int nchunks,
                                                     const double *__restrict__ partials, double *__restrict__ G,
                                                     const double *colsum, const double *Aold, double *A,
                                                     NnlsParams *prm) {
  const int lane = threadIdx.x & 63;           // (R <= 64; the column sums are sums of magnitudes)
  const bool hit = __ballot(lane < R && colsum[lane] == 0.0) != 0ull;
  if (blockIdx.x == 0 && threadIdx.x == 0) prm->fallback = hit;
  if (!hit) {
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < R * R; e += gridDim.x * blockDim.x)
      G[e] = combine_chunks(partials, e, R * R, nchunks);
    return;
  }
  if (blockIdx.x != 0) return;
  for (int e = threadIdx.x; e < R * R; e += blockDim.x) {
    const int a = e / R, b = e % R;
    double g = 0.0;
    for (int c = 0; c < nchunks; ++c) {
      double p = 0.0;
      for (int64_t i = 32 * (int64_t)c; i < I && i < 32 * (int64_t)(c + 1); ++i)
        p = fma(zero_col_mix(A[i * ldr + a], Aold[i * ldr + a]), zero_col_mix(A[i * ldr + b], Aold[i * ldr + b]), p);
      g = c == 0 ? p : g + p;
    }
    G[e] = g;
  }
  __syncthreads();                            // every entry of G read A before it changes
  const int c = threadIdx.x & 63;
  if (c >= R) return;
  for (int64_t row = threadIdx.x >> 6; row < I; row += blockDim.x >> 6) {
    const int64_t e = row * ldr + c;
    A[e] = zero_col_mix(A[e], Aold[e]);
  }
}

// <M, A> over I x ldr (padding is zero in both) and <V, G> over R x R: per-thread
// strided partial sums, then a fixed-shape tree in LDS (deterministic).  The Gram-form
// cost sqrt(||X||^2 - 2<M,A> + <V,G>) (CpdCUDA.hpp:137-142) or, for the accelerated
// factors, sqrt(||X||^2 + <V,G> - 2<M,A>) (Cpd.hpp:162-169).
__global__ __launch_bounds__(1024) void k_cost_gram(int64_t nma, const double *__restrict__ M,
                                                    const double *__restrict__ A, int R, const double *__restrict__ V,
                                                    const double *__restrict__ G, const double *frob, double *f,
                                                    int accel) {
  __shared__ double rma[1024], rvg[1024];
  const int tid = threadIdx.x;
  double ma = 0.0, vg = 0.0;
  for (int64_t e = tid; e < nma; e += 1024) ma = fma(M[e], A[e], ma);
  for (int e = tid; e < R * R; e += 1024) vg = fma(V[e], G[e], vg);
  rma[tid] = ma;
  rvg[tid] = vg;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if (tid < w) {
      rma[tid] += rma[tid + w];
      rvg[tid] += rvg[tid + w];
    }
    __syncthreads();
  }
  if (tid == 0) *f = accel ? sqrt(*frob + rvg[0] - 2.0 * rma[0]) : sqrt(*frob - 2.0 * rma[0] + rvg[0]);
}

// Normalize (Normalize.hpp:92-174): factors 0..N-2 other than the weight factor wf are
// scaled to unit columns, wf absorbs the product of their norms, the last factor is
// never touched and the zero test reads only the last lambda_fac entry; the Grams are
// rescaled by quotients.
struct NormArgs {
  int N, R, ldr, wf;
  int64_t dims[kMaxOrder];
  double *G[kMaxOrder];
  double *A[kMaxOrder];
};

// Column norms, scales and the Gram rescaling of Normalize (one block).  Columns whose
// norms vanish keep scale 1 on every factor, so the row pass leaves them bit-identical.
// After every thread of the block has stored its part of a readback to mapped host
// memory: one thread fences at system scope and stores the sequence word (vector store).
__device__ __forceinline__ void publish_seq(unsigned *dst, unsigned seq) {
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence_system();
    *(volatile unsigned *)dst = seq;
  }
}

__global__ __launch_bounds__(256) void k_normalize(NormArgs na, double *scratch, ExportList ex) {
  // the sweep's readback first (it does not depend on Normalize)
  for (int q = 0; q < ex.count; ++q)
    for (int e = threadIdx.x; e < ex.words[q]; e += blockDim.x) ex.dst[q][e] = ex.src[q][e];
  if (ex.seq_dst) publish_seq(ex.seq_dst, ex.seq);
  const int N = na.N, R = na.R, last = N - 1;
  double *lam = scratch;                       // (N-1) x R
  double *scale = scratch + kMaxOrder * kMaxRank;  // N x R column scales (1 = untouched)
  if (threadIdx.x < R) {
    const int i = threadIdx.x;
    int pass = 0;
    for (int k = 0; k < N; ++k) {
      if (k != na.wf) lam[(k - pass) * R + i] = na.G[k][i * R + i];
      else pass = 1;
      scale[k * R + i] = 1.0;
    }
    double nf[kMaxOrder];
    int nz = 1;
    for (int j = 0; j < last; ++j) {
      nf[j] = sqrt(lam[j * R + i]);
      nz = !(nf[j] == 0.0);
    }
    if (!nz) {
      for (int j = 0; j < last; ++j) lam[j * R + i] = 1.0;
    } else {
      double cumul = 1.0;
      pass = 0;
      for (int j = 0; j < last; ++j) {
        if (j == na.wf) { pass = 1; continue; }
        scale[j * R + i] = 1.0 / nf[j - pass];
        cumul *= nf[j - pass];
        lam[(j - pass) * R + i] = nf[j - pass];
      }
      scale[na.wf * R + i] = cumul;
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < R * R; e += blockDim.x) {
    int a = e / R, b = e % R;
    double nmw = 1.0;
    int pass = 0;
    for (int i = 0; i < last; ++i) {
      if (i == na.wf) { pass = 1; continue; }
      const double *l = lam + (i - pass) * R;
      double nm = l[a] * l[b];
      nmw = nmw * nm;
      na.G[i][e] = na.G[i][e] / nm;
    }
    na.G[na.wf][e] = na.G[na.wf][e] * nmw;
  }
}

// Row pass of Normalize: A_k[row][c] *= scale[k][c]; block (row tile of 4, factor k).
// With ax.out the line-search step of k_axpy_accel follows for every entry of the row
// (padding included): A_hat = A_old + step (A - A_old), A_old = A, snap = A.
__global__ __launch_bounds__(256) void k_normalize_rows(NormArgs na, const double *__restrict__ scratch,
                                                        AxpyArgs ax) {
  const int k = blockIdx.y, c = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= na.dims[k]) return;
  const bool scaled = !(k == na.N - 1 && k != na.wf) && c < na.R;
  double *a = na.A[k] + row * na.ldr + c;
  if (!ax.out) {
    if (scaled) *a = *a * scratch[kMaxOrder * kMaxRank + k * na.R + c];
    return;
  }
  if (c >= na.ldr) return;
  double v = *a;
  if (scaled) {
    v = v * scratch[kMaxOrder * kMaxRank + k * na.R + c];
    *a = v;
  }
  const double step = (ax.coeff == nullptr || *ax.coeff == ax.c) ? ax.step_c : ax.step_c1;
  const int64_t e = (na.A[k] - ax.cur) + row * na.ldr + c;
  const double o = ax.old[e];
  ax.out[e] = o + step * (v - o);
  ax.old[e] = v;
  if (ax.snap) ax.snap[e] = v;
}

// A_hat = A_old + step (A - A_old) (Cpd.hpp:251-258).  The step depends on the current
// acceleration coefficient, which the device updates: step_c for *coeff == c, else
// step_c1 (the coefficient rises by at most one per sweep).
// The same pass sets A_old = A for the next sweep (Cpd.hpp:348,353) and, when snap is
// given, copies A there too.
__global__ void k_axpy_accel(int64_t n, double step_c, double step_c1, int c, const int *coeff, double *old,
                             const double *cur, double *out, double *snap) {
  const double step = (coeff == nullptr || *coeff == c) ? step_c : step_c1;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const double o = old[e], a = cur[e];
    out[e] = o + step * (a - o);
    old[e] = a;
    if (snap) snap[e] = a;
  }
}

// Small device-to-host copies in one launch (4-byte words; dst is mapped host memory).
__global__ void k_export(ExportList x) {
  for (int q = 0; q < x.count; ++q)
    for (int e = threadIdx.x; e < x.words[q]; e += blockDim.x) x.dst[q][e] = x.src[q][e];
  if (x.seq_dst) publish_seq(x.seq_dst, x.seq);
}

// Line-search decision on the device (Cpd.hpp:262-269): accept the accelerated factors
// when f > f_hat, unless the run stops on the threshold at this sweep (the reference
// checks termination first, Cpd.hpp:339-346).  On acceptance the accelerated factors,
// their Grams and the mode-0 NNLS set-up prepared for them replace the current ones.
// flags[0] = accepted, flags[1] = threshold stop, flags[2] / flags[3] = accel_fail /
// accel_coeff, kept as line_search_accel keeps them (Cpd.hpp:270-277).
__global__ void k_accel_decide(const double *__restrict__ scal, double thr, int *flags, AccelCopy cp) {
  const double f = scal[1], fa = scal[2];
  const bool stop = f / sqrt(scal[0]) < thr;
  const bool accept = !stop && f > fa;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    flags[0] = accept ? 1 : 0;
    flags[1] = stop ? 1 : 0;
    if (!stop) {
      int fail = flags[2] + (accept ? 0 : 1);
      if (fail == 5) {
        fail = 0;
        flags[3] = flags[3] + 1;
      }
      flags[2] = fail;
    }
    if (cp.fa_out) {
      *cp.fa_out = fa;
      for (int q = 0; q < 4; ++q) cp.flags_out[q] = flags[q];
    }
    if (cp.f_out) *cp.f_out = f;
    if (cp.seq_dst) {                        // the sweep's readback is complete
      __threadfence_system();
      *(volatile unsigned *)cp.seq_dst = cp.seq;
    }
  }
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  if (cp.pick_n) {
    const double *src = accept ? cp.pick_src[0] : cp.pick_src[1];
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < cp.pick_n; e += stride)
      cp.pick_dst[e] = src[e];
  }
  if (!accept) return;
  for (int q = 0; q < 4; ++q)
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < cp.n[q]; e += stride)
      cp.dst[q][e] = cp.src[q][e];
  if (cp.prm_src && blockIdx.x == 0 && threadIdx.x == 0) *cp.prm_dst = *cp.prm_src;
}

int grid_for(int64_t n, int block) {
  int64_t g = (n + block - 1) / block;
  if (g > 65536) g = 65536;
  if (g < 1) g = 1;
  return (int)g;
}

}  // namespace

void hadamard(hipStream_t s, int R, int ng, const double *const *grams, double *V) {
  GramPtrs G{};
  for (int j = 0; j < ng; ++j) G.p[j] = grams[j];
  k_hadamard<<<1, 256, 0, s>>>(R, ng, G, V);
}

void gram(hipStream_t s, int64_t I, int R, int ldr, const double *A, double *G, double *partials) {
  const int nchunks = (int)((I + 31) / 32);
#define PTN_GC(NTV) \
  if (ldr == 16 * NTV) k_gram_chunks<NTV><<<nchunks, 256, 0, s>>>(I, R, A, partials)
  PTN_GC(1);
  PTN_GC(2);
  PTN_GC(3);
  PTN_GC(4);
#undef PTN_GC
  k_gram_combine<<<(unsigned)((R * R + 63) / 64), 64, 0, s>>>(R, nchunks, partials, G);
}

void grams_all(hipStream_t s, int N, const int64_t *dims, int R, int ldr, const double *const *A, double *const *G,
               int ng, const int *list, double *V, double *partials) {
  GramBatch b{};
  b.N = N;
  b.ng = ng;
  for (int k = 0; k < N; ++k) {
    b.I[k] = dims[k];
    b.A[k] = A[k];
    b.G[k] = G[k];
    b.chunk0[k + 1] = b.chunk0[k] + (int)((dims[k] + 31) / 32);
  }
  for (int j = 0; j < ng; ++j) b.list[j] = list[j];
#define PTN_GA(NTV) \
  if (ldr == 16 * NTV) k_gram_chunks_all<NTV><<<(unsigned)b.chunk0[N], 256, 0, s>>>(b, R, partials)
  PTN_GA(1);
  PTN_GA(2);
  PTN_GA(3);
  PTN_GA(4);
#undef PTN_GA
  k_gram_combine_all<<<(unsigned)((R * R + 63) / 64), 64 * N, 0, s>>>(b, R, partials, V);
}

void eig_extremes(hipStream_t s, int R, const double *V, NnlsParams *p, int max_inner, double *betas) {
  const GramPtrs G{};
  if (R <= 16) k_eig_extremes<16><<<1, kEigThreads<16>, 0, s>>>(R, V, G, 0, nullptr, p, max_inner, betas);
  else if (R <= 32) k_eig_extremes<32><<<1, kEigThreads<32>, 0, s>>>(R, V, G, 0, nullptr, p, max_inner, betas);
  else k_eig_extremes<64><<<1, kEigThreads<64>, 0, s>>>(R, V, G, 0, nullptr, p, max_inner, betas);
}

void nnls_setup(hipStream_t s, int R, int ng, const double *const *grams, double *V, NnlsParams *p, int max_inner,
                double *betas) {
  GramPtrs G{};
  for (int j = 0; j < ng; ++j) G.p[j] = grams[j];
  if (R <= 16) k_eig_extremes<16><<<1, kEigThreads<16>, 0, s>>>(R, nullptr, G, ng, V, p, max_inner, betas);
  else if (R <= 32) k_eig_extremes<32><<<1, kEigThreads<32>, 0, s>>>(R, nullptr, G, ng, V, p, max_inner, betas);
  else k_eig_extremes<64><<<1, kEigThreads<64>, 0, s>>>(R, nullptr, G, ng, V, p, max_inner, betas);
}

void nnls_iterate(hipStream_t s, int64_t I, int R, int ldr, const double *V, const NnlsParams *p,
                  const double *betas, const double *M, const double *A, const double *S, double d1, double d2,
                  int max_inner, uint64_t *mask, double *hist, double *colsum) {
  const unsigned grid = (unsigned)((I + 3) / 4);
  unsigned long long *m = (unsigned long long *)mask;
#define PTN_NI(RBV) \
  k_nnls_iterate<RBV><<<grid, 256, 0, s>>>(I, R, ldr, V, p, betas, M, A, S, d1, d2, max_inner, m, hist, colsum)
  if (R <= 16) PTN_NI(16);
  else if (R <= 32) PTN_NI(32);
  else PTN_NI(64);
#undef PTN_NI
}

void nnls_finish(hipStream_t s, int64_t I, int R, int ldr, const double *hist, const uint64_t *mask, int max_inner,
                 double *A, double *colsum, const double *Aold, double *G, double *partials, NnlsParams *p) {
  const int nchunks = (int)((I + 31) / 32);
#define PTN_NF(NTV)                                                                                         \
  if (ldr == 16 * NTV)                                                                                      \
  k_nnls_finish<NTV><<<(unsigned)nchunks, 256, 0, s>>>(I, R, hist, (const unsigned long long *)mask, max_inner, A, \
                                                       colsum, partials, p)
  PTN_NF(1);
  PTN_NF(2);
  PTN_NF(3);
  PTN_NF(4);
#undef PTN_NF
  k_gram_finish<<<(unsigned)((R * R + 255) / 256), 256, 0, s>>>(I, R, ldr, nchunks, partials, G, colsum, Aold, A, p);
}

void nnls_select(hipStream_t s, int64_t I, int R, int ldr, const double *hist, const uint64_t *mask, int max_inner,
                 double *Anew, double *colsum, NnlsParams *p) {
  int64_t g = (I + 3) / 4;
  if (g > 256) g = 256;
  k_nnls_select<<<(unsigned)g, 256, 0, s>>>(I, R, ldr, hist, (const unsigned long long *)mask, max_inner, Anew,
                                            colsum, p);
}

void cost_gram(hipStream_t s, int64_t nma, const double *M, const double *A, int R, const double *V, const double *G,
               const double *frob, double *f, int accel) {
  k_cost_gram<<<1, 1024, 0, s>>>(nma, M, A, R, V, G, frob, f, accel);
}

void normalize(hipStream_t s, int N, const int64_t *dims, int R, int ldr, int wf, double *const *grams,
               double *const *fac, double *scratch, const ExportList *ex, const AxpyArgs *ax) {
  NormArgs na{};
  na.N = N; na.R = R; na.ldr = ldr; na.wf = wf;
  for (int k = 0; k < N; ++k) { na.dims[k] = dims[k]; na.G[k] = grams[k]; na.A[k] = fac[k]; }
  int64_t maxI = 0;
  for (int k = 0; k < N; ++k) maxI = dims[k] > maxI ? dims[k] : maxI;
  ExportList e0{};
  AxpyArgs a0{};
  k_normalize<<<1, 256, 0, s>>>(na, scratch, ex ? *ex : e0);
  k_normalize_rows<<<dim3((unsigned)((maxI + 3) / 4), (unsigned)N), 256, 0, s>>>(na, scratch, ax ? *ax : a0);
}

void accel_decide(hipStream_t s, const double *scal, double thr, int *flags, const AccelCopy &cp) {
  k_accel_decide<<<grid_for(cp.n[0] > 4096 ? cp.n[0] : 4096, 256), 256, 0, s>>>(scal, thr, flags, cp);
}

void axpy_accel(hipStream_t s, int64_t n, double step_c, double step_c1, int c, const int *coeff, double *old,
                const double *cur, double *out, double *snap) {
  k_axpy_accel<<<grid_for(n, 256), 256, 0, s>>>(n, step_c, step_c1, c, coeff, old, cur, out, snap);
}

void export_words(hipStream_t s, const ExportList &x) { k_export<<<1, 256, 0, s>>>(x); }

}  // namespace ptn
