// The learned NNLS warm start: a 3-layer MLP (2208 -> 256 -> 256 -> 64, ReLU) that maps
// one factor row's subproblem (the Gram V, the MTTKRP row, the previous row) to a start
// point for NesterovMNLS.  BF16 weights and activations, FP32 accumulation on
// v_mfma_f32_32x32x16_bf16, FP32 master weights updated by Adam.  The subproblem itself is
// never changed: the network only proposes the start, the proximal anchor stays the
// previous factor row, and a row keeps the previous row as its start unless the proposal
// passes the KKT test in k_warm_select.
#include "ptn_internal.hpp"

namespace ptn {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// ---------------------------------------------------------------------------
// C[m][n] = sum_k A[m][k] B[n][k] (+ bias[n]) (* (gate[m][n] > 0)) (ReLU), both operands
// bf16 with k contiguous (K a multiple of 16, leading dimensions multiples of 8).  A block
// is one wave with a 32 x 32 tile.  Rows / columns past M / N read a clamped row and are
// not stored.  Cbt: a transposed copy of the bf16 result (ldcbt a multiple of 4), so that
// the weight gradients find their operands k-contiguous.
//
// The layers are small, so neither the matrix cores nor the memory bound them but a wave's
// loads: fetching the fragments where they lie takes 64 cache lines for each load, and four
// waves to a block left three CUs in four idle at 1024 rows.  So a wave fetches 128 k of its
// 64 rows with sixteen lanes to a row, two such groups in flight, and takes the fragments from
// LDS (rows 272 bytes apart: sixteen rows lie in different banks).  Average over the eight
// products of a step of 1024 rows: 15.0 us, with the two groups but fragments fetched where they
// lie 14.1 us, so 8.9 us.
// ---------------------------------------------------------------------------
struct GemmNt {
  int M, N, K, lda, ldb, ldg, relu, ldc, ldcb, ldcbt;
  const __bf16 *A, *B;
  const float *bias;
  const __bf16 *gate;
  float *C;
  __bf16 *Cb, *Cbt;
  __host__ __device__ int tiles_n() const { return (N + 31) / 32; }
  __host__ __device__ int tiles() const { return tiles_n() * ((M + 31) / 32); }
};
constexpr int kGemmLd = 128 + 8, kGemmLds = 64 * kGemmLd * 2;   // bytes: 32 rows of A, 32 of B
__device__ __forceinline__ void gemm_tile(const GemmNt &g, int b, __bf16 *tile) {
  const int M = g.M, N = g.N, K = g.K, lda = g.lda, ldb = g.ldb;
  const __bf16 *__restrict__ A = g.A, *__restrict__ B = g.B, *__restrict__ gate = g.gate;
  const float *__restrict__ bias = g.bias;
  float *__restrict__ C = g.C;
  __bf16 *__restrict__ Cb = g.Cb, *__restrict__ Cbt = g.Cbt;
  constexpr int KG = 128, LD = kGemmLd;
  const int lane = threadIdx.x, i = lane & 31, kg = lane >> 5;
  const int m0 = b / g.tiles_n() * 32, n0 = b % g.tiles_n() * 32;
  const int fr = lane >> 4, fc = 8 * (lane & 15);        // fetching: row within four, first column
  const __bf16 *pa[8], *pb[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int m = m0 + 4 * q + fr, n = n0 + 4 * q + fr;
    pa[q] = A + (int64_t)(m < M ? m : M - 1) * lda;
    pb[q] = B + (int64_t)(n < N ? n : N - 1) * ldb;
  }
  struct Rows {
    bf16x8 a[8], b[8];
  };
  auto load = [&](int k, Rows &f) {
    const int c = k + fc < K ? k + fc : 0;               // a column past K: read, never used
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      f.a[q] = *(const bf16x8 *)(pa[q] + c);
      f.b[q] = *(const bf16x8 *)(pb[q] + c);
    }
  };
  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f;
  auto mul = [&](int k, const Rows &f, Rows &next) {     // then group k + 2 KG into next
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      *(bf16x8 *)(tile + (4 * q + fr) * LD + fc) = f.a[q];
      *(bf16x8 *)(tile + (32 + 4 * q + fr) * LD + fc) = f.b[q];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (k + 2 * KG < K) load(k + 2 * KG, next);
    const __bf16 *ta = tile + i * LD + 8 * kg, *tb = ta + 32 * LD;
    const int nu = K - k < KG ? (K - k) / 16 : KG / 16;
#pragma unroll
    for (int u = 0; u < KG / 16; ++u)
      if (u < nu)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8 *)(ta + 16 * u), *(const bf16x8 *)(tb + 16 * u),
                                                      acc, 0, 0, 0);
  };
  Rows f0, f1;
  load(0, f0);
  if (KG < K) load(KG, f1);
  for (int k = 0; k < K; k += 2 * KG) {
    mul(k, f0, f0);
    if (k + KG < K) mul(k + KG, f1, f1);
  }
  const int n = n0 + i;
  if (n >= N) return;
  const float bn = bias ? bias[n] : 0.f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    bf16x4 t4;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + 8 * q + 4 * kg + r;
      float x = acc[4 * q + r] + bn;
      if (m < M) {
        if (gate && !((float)gate[(int64_t)m * g.ldg + n] > 0.f)) x = 0.f;
        if (g.relu) x = x > 0.f ? x : 0.f;
        if (C) C[(int64_t)m * g.ldc + n] = x;
        if (Cb) Cb[(int64_t)m * g.ldcb + n] = (__bf16)x;
      }
      t4[r] = (__bf16)x;
    }
    // (M is a multiple of 4 wherever a transposed copy is asked for)
    if (Cbt && m0 + 8 * q + 4 * kg < M) *(bf16x4 *)(Cbt + (int64_t)n * g.ldcbt + m0 + 8 * q + 4 * kg) = t4;
  }
}

// Several transposes in one launch: out[c][r] = in[r][c] (bf16), 32 x 32 tiles through LDS; block b
// belongs to the matrix whose tiles start at or before b.  (Eight launches of 4.7 us a step of an
// epoch of 8192 rows in batches of 1024; the layers' own results are written transposed by their
// products.)
struct Transposes {
  int n;
  int first[5];                                         // first tile of each matrix, then their number
  int rows[4], cols[4], ldi[4], ldo[4];
  const __bf16 *in[4];
  __bf16 *out[4];
};
__global__ __launch_bounds__(256) void k_transposes(Transposes T) {
  __shared__ __bf16 t[32][33];
  int w = 0;
  while (w + 1 < T.n && (int)blockIdx.x >= T.first[w + 1]) ++w;
  const int tile = blockIdx.x - T.first[w], tc = (T.cols[w] + 31) / 32;
  const int r0 = tile / tc * 32, c0 = tile % tc * 32, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int rows = T.rows[w], cols = T.cols[w];
  const __bf16 *in = T.in[w];
  __bf16 *out = T.out[w];
#pragma unroll
  for (int y = ty; y < 32; y += 8) {
    const int r = r0 + y, c = c0 + tx;
    t[y][tx] = (r < rows && c < cols) ? in[(int64_t)r * T.ldi[w] + c] : (__bf16)0.f;
  }
  __syncthreads();
#pragma unroll
  for (int y = ty; y < 32; y += 8) {
    const int c = c0 + y, r = r0 + tx;
    if (c < cols && r < rows) out[(int64_t)c * T.ldo[w] + r] = t[tx][y];
  }
}

// ---------------------------------------------------------------------------
// Features of factor rows (one 64-lane wave per row, lane = column c < 64):
//   [ vech(V) / sV (upper triangle of the 64 x 64 zero-padded V, row by row),
//     m / s_m, a_prev * sV / s_m ],   sV = max_k V_kk, s_m = max_c |m_c| (1 if 0).
// The target of a solution row a* is a* sV / s_m.  scale[row] = s_m / sV maps the
// network's output back.  With Anew: targets T[row][c] (zero beyond R) and rank[row] = R.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int vech_index(int a, int b) {       // a <= b < 64
  return a * kMlpR - (a * (a - 1)) / 2 + (b - a);
}

__global__ __launch_bounds__(256) void k_mlp_features(int64_t I, int R, int ldr, const double *__restrict__ V,
                                                      const double *__restrict__ M, const double *__restrict__ A,
                                                      const double *__restrict__ Anew, __bf16 *__restrict__ X,
                                                      float *__restrict__ T, unsigned char *__restrict__ rank,
                                                      float *__restrict__ scale) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= I) return;
  double sv = 0.0;
  for (int k = 0; k < R; ++k) sv = fmax(sv, V[k * R + k]);
  if (!(sv > 0.0)) sv = 1.0;
  const bool on = lane < R;
  const double m = on ? M[row * ldr + lane] : 0.0;
  double sm = fabs(m);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sm = fmax(sm, __shfl_xor(sm, o, 64));
  if (!(sm > 0.0)) sm = 1.0;
  __bf16 *x = X + row * kMlpIn;
  // lane c writes row c of the upper triangle: entries (c, c..63)
  for (int b = lane; b < kMlpR; ++b) {
    const double v = (lane < R && b < R) ? V[lane * R + b] / sv : 0.0;
    x[vech_index(lane, b)] = (__bf16)(float)v;
  }
  x[kMlpVech + lane] = (__bf16)(float)(m / sm);
  x[kMlpVech + kMlpR + lane] = (__bf16)(float)(on ? A[row * ldr + lane] * sv / sm : 0.0);
  if (scale && lane == 0) scale[row] = (float)(sm / sv);
  if (T) T[row * kMlpR + lane] = (float)(on ? Anew[row * ldr + lane] * sv / sm : 0.0);
  if (rank && lane == 0) rank[row] = (unsigned char)R;
}

// ---------------------------------------------------------------------------
// The warm-start decision (one wave per row, lane = column).  With Zt = V + lambda I,
// wt = m + lambda a_prev (the subproblem NesterovMNLS solves, anchor unchanged) and L its
// Lipschitz constant, the relative KKT residual of a start a is the projected-gradient
// fixed-point residual min(a, g / L), g = a Zt - wt, relative to the solution's scale
// max|wt| / L:  r(a) = max_c |min(L a_c, g_c)| / max_c |wt_c|.
// The row starts from the network's proposal a_p = max(y, 0) * scale when y is finite and
// r(a_p) <= kkt_tol; otherwise from a_prev (the fallback, which is exactly the reference's
// start).  With C, the proposal is C's row instead (max(C, 0): the proposals after some
// Nesterov steps, whose count, prm->iters, is kept in prm->warm_steps).  S receives the
// start rows (S may be C); count, when given, the rows that took the proposal.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_warm_select(int64_t I, int R, int ldr, const double *__restrict__ V,
                                                     NnlsParams *prm, const double *__restrict__ M,
                                                     const double *__restrict__ A, const float *__restrict__ Y,
                                                     const float *__restrict__ scale, const double *C,
                                                     double kkt_tol, double *S, int *count) {
  if (C && blockIdx.x == 0 && threadIdx.x == 0) prm->warm_steps = prm->iters;
  __shared__ double buf[4][kMlpR];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave;
  if (row >= I) return;
  const bool on = lane < R;
  const double lambda = prm->lambda, L = prm->L;
  const double ap = on ? A[row * ldr + lane] : 0.0;
  bool fin;
  double aw;
  if (C) {
    const double c = on ? C[row * ldr + lane] : 0.0;
    fin = !on || isfinite(c);
    aw = c > 0.0 ? c : 0.0;
  } else {
    const float y = on ? Y[row * kMlpR + lane] : 0.f;
    fin = !on || isfinite(y);
    aw = (on && y > 0.f) ? (double)y * (double)scale[row] : 0.0;
  }
  buf[wave][lane] = aw;
  __builtin_amdgcn_wave_barrier();
  double gw = 0.0;
  if (on) {
    for (int k = 0; k < R; ++k) {
      const double z = V[k * R + lane] + (k == lane ? lambda : 0.0);
      gw = fma(buf[wave][k], z, gw);
    }
  }
  const double wt = on ? M[row * ldr + lane] + lambda * ap : 0.0;
  gw -= wt;
  double rw = fabs(fmin(L * aw, gw)), sw = fabs(wt);
  if (!on) rw = sw = 0.0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    rw = fmax(rw, __shfl_xor(rw, o, 64));
    sw = fmax(sw, __shfl_xor(sw, o, 64));
  }
  const bool all_fin = __ballot(!fin) == 0ull;
  const double den = sw > 0.0 ? sw : 1.0;
  const bool take = all_fin && rw / den <= kkt_tol;
  if (lane < ldr) S[row * ldr + lane] = take ? (on ? aw : 0.0) : (lane < R ? ap : A[row * ldr + lane]);
  if (count && take && lane == 0) atomicAdd(count, 1);
}

// loss = sum over valid entries (c < rank[row]) of (Y - T)^2 / count; dY = 2 (Y - T) / count
// (bf16 for the weight gradient, FP32 for the bias gradient); partial sums per block.
__global__ __launch_bounds__(256) void k_mse_grad(int B, const float *__restrict__ Y, const float *__restrict__ T,
                                                  const unsigned char *__restrict__ rank, float inv_count,
                                                  __bf16 *__restrict__ dYb, float *__restrict__ dY,
                                                  double *__restrict__ part) {
  __shared__ double red[256];
  const int64_t n = (int64_t)B * kMlpR;
  double s = 0.0;
  for (int64_t e = blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
    const int64_t r = e / kMlpR;
    const int c = (int)(e - r * kMlpR);
    float g = 0.f;
    if (c < rank[r]) {
      const float d = Y[e] - T[e];
      s += (double)d * d;
      g = 2.f * d * inv_count;
    }
    dYb[e] = (__bf16)g;
    dY[e] = g;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0] * inv_count;
}

// Bias gradient: out[n] = sum_m G[m][n] (FP32 or bf16 rows), rows added in order in FP32: a chain
// of M dependent adds per column, which bounds it.  A block owns 16 columns (N and ldg are
// multiples of 16, rows 16-byte aligned): its 64 threads fetch 256 rows at a time with 16-byte
// loads, four rows each, and leave them column by column in LDS, where 16 lanes walk their columns
// four rows per read while the next 256 rows are on their way.  One thread per column reading
// its rows from memory one by one waited for every load: 1024 rows of 256 columns 224 us, so
// 6.4 us (an epoch of 8192 rows in batches of 1024: 7.2 -> 1.9 ms).  Rows past M enter as +0,
// which leaves a sum that starts at +0 as it is.
struct Colsum {
  int M, N, ldg;
  const void *G;
  float *out;
  __host__ __device__ int tiles() const { return N / 16; }
};
constexpr int kColsumLd = 256 + 4, kColsumLds = 16 * kColsumLd * 4;   // 16 lanes x 16-byte reads touch every bank once
template <typename TG>
__device__ __forceinline__ void colsum_tile(const Colsum &cs, int b, float *tile) {
  constexpr int LD = kColsumLd;
  typedef TG v8 __attribute__((ext_vector_type(16 / sizeof(TG))));
  constexpr int NV = 16 * sizeof(TG) / 16;      // 16-byte loads per row
  const int M = cs.M, ldg = cs.ldg, t = threadIdx.x, n0 = b * 16;
  const TG *G = (const TG *)cs.G;
  v8 pre[4][NV];
  auto fetch = [&](int m0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int m = m0 + 64 * u + t;
      const v8 *p = (const v8 *)(G + (int64_t)(m < M ? m : M - 1) * ldg + n0);
#pragma unroll
      for (int q = 0; q < NV; ++q) pre[u][q] = p[q];
    }
  };
  float s = 0.f;
  fetch(0);
  for (int m0 = 0; m0 < M; m0 += 256) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool in = m0 + 64 * u + t < M;
#pragma unroll
      for (int c = 0; c < 16; ++c)
        tile[c * LD + 64 * u + t] = in ? (float)pre[u][c / (16 / NV)][c % (16 / NV)] : 0.f;
    }
    __syncthreads();
    if (m0 + 256 < M) fetch(m0 + 256);
    if (t < 16) {
      const float4 *p = (const float4 *)(tile + t * LD);
#pragma unroll 16
      for (int r = 0; r < 64; ++r) {
        const float4 v = p[r];
        s += v.x;
        s += v.y;
        s += v.z;
        s += v.w;
      }
    }
  }
  if (t < 16) cs.out[n0 + t] = s;
}

// One launch for what a step can do at once: the column sums' blocks first (the longest chain),
// then the tiles of up to two products.  Each fills a part of the chip for 5 to 9 us, so their
// launches one after the other were half of a backward pass (epoch as above: 1251 -> 987 us).
template <typename TG>
__global__ __launch_bounds__(64) void k_layers(Colsum cs, GemmNt g0, GemmNt g1) {
  __shared__ __align__(16) unsigned char lds[kGemmLds > kColsumLds ? kGemmLds : kColsumLds];
  int b = blockIdx.x;
  const int nc = cs.tiles();
  if (b < nc) {
    colsum_tile<TG>(cs, b, (float *)lds);
    return;
  }
  b -= nc;
  if (b < g0.tiles()) gemm_tile(g0, b, (__bf16 *)lds);
  else gemm_tile(g1, b - g0.tiles(), (__bf16 *)lds);
}

// Adam (Kingma & Ba 2015) on the FP32 master weights; the bf16 copies of the three weight
// matrices follow (the biases are used in FP32).
__global__ void k_adam(int64_t n, float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m1,
                       float *__restrict__ m2, float lr, float b1, float b2, float eps, float c1, float c2,
                       __bf16 *__restrict__ wb) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const float gr = g[e];
    const float a = b1 * m1[e] + (1.f - b1) * gr;
    const float b = b2 * m2[e] + (1.f - b2) * gr * gr;
    m1[e] = a;
    m2[e] = b;
    const float x = w[e] - lr * (a * c1) / (sqrtf(b * c2) + eps);
    w[e] = x;
    const int64_t bi = mlp_bf16_index(e);
    if (bi >= 0) wb[bi] = (__bf16)x;
  }
}

// bf16 copies of the weight matrices from the FP32 master vector
__global__ void k_weights_bf16(int64_t n, const float *__restrict__ w, __bf16 *__restrict__ wb) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t bi = mlp_bf16_index(e);
    if (bi >= 0) wb[bi] = (__bf16)w[e];
  }
}

// rows idx[0..B) of a data set into contiguous batch buffers (X bf16, T FP32, rank)
__global__ __launch_bounds__(256) void k_gather(int B, const int *__restrict__ idx, const __bf16 *__restrict__ X,
                                                const float *__restrict__ T, const unsigned char *__restrict__ rank,
                                                __bf16 *__restrict__ Xb, float *__restrict__ Tb,
                                                unsigned char *__restrict__ rb) {
  const int r = blockIdx.x;
  if (r >= B) return;
  const int64_t src = idx[r];
  const uint4 *xs = (const uint4 *)(X + src * kMlpIn);
  uint4 *xd = (uint4 *)(Xb + (int64_t)r * kMlpIn);
  for (int e = threadIdx.x; e < kMlpIn / 8; e += blockDim.x) xd[e] = xs[e];
  if (threadIdx.x < kMlpR) Tb[(int64_t)r * kMlpR + threadIdx.x] = T[src * kMlpR + threadIdx.x];
  if (threadIdx.x == 0) rb[r] = rank[src];
}

}  // namespace

namespace {
GemmNt gemm_args(const LayerProduct &p) {
  return GemmNt{p.M, p.N, p.K, p.lda, p.ldb, p.ldg, p.relu, p.ldc, p.ldcb, p.ldcbt, (const __bf16 *)p.A,
                (const __bf16 *)p.B, p.bias, (const __bf16 *)p.gate, p.C, (__bf16 *)p.Cb, (__bf16 *)p.Cbt};
}
}  // namespace

void layer_products(hipStream_t s, const LayerProduct &p0, const LayerProduct *p1, const ColumnSums *sums) {
  const GemmNt g0 = gemm_args(p0), g1 = p1 ? gemm_args(*p1) : GemmNt{};
  const Colsum cs = sums ? Colsum{sums->M, sums->N, sums->N, sums->G, sums->out} : Colsum{};
  const unsigned grid = (unsigned)(cs.tiles() + g0.tiles() + g1.tiles());
  if (sums && sums->f32) k_layers<float><<<grid, 64, 0, s>>>(cs, g0, g1);
  else k_layers<__bf16><<<grid, 64, 0, s>>>(cs, g0, g1);
}

void transposes_bf16(hipStream_t s, int n, const TransposeBf16 *m) {
  Transposes T{};
  T.n = n;
  for (int w = 0; w < n; ++w) {
    T.rows[w] = m[w].rows;
    T.cols[w] = m[w].cols;
    T.ldi[w] = m[w].cols;
    T.ldo[w] = m[w].rows;
    T.in[w] = (const __bf16 *)m[w].in;
    T.out[w] = (__bf16 *)m[w].out;
    T.first[w + 1] = T.first[w] + (m[w].rows + 31) / 32 * ((m[w].cols + 31) / 32);
  }
  k_transposes<<<T.first[n], 256, 0, s>>>(T);
}

void mlp_features(hipStream_t s, int64_t I, int R, int ldr, const double *V, const double *M, const double *A,
                  const double *Anew, void *X, float *T, unsigned char *rank, float *scale) {
  k_mlp_features<<<(unsigned)((I + 3) / 4), 256, 0, s>>>(I, R, ldr, V, M, A, Anew, (__bf16 *)X, T, rank, scale);
}

void warm_select(hipStream_t s, int64_t I, int R, int ldr, const double *V, NnlsParams *p, const double *M,
                 const double *A, const float *Y, const float *scale, const double *C, double kkt_tol, double *S,
                 int *count) {
  k_warm_select<<<(unsigned)((I + 3) / 4), 256, 0, s>>>(I, R, ldr, V, p, M, A, Y, scale, C, kkt_tol, S, count);
}

void mse_grad(hipStream_t s, int B, const float *Y, const float *T, const unsigned char *rank, float inv_count,
              void *dYb, float *dY, double *part, int nparts) {
  k_mse_grad<<<nparts, 256, 0, s>>>(B, Y, T, rank, inv_count, (__bf16 *)dYb, dY, part);
}

void adam_step(hipStream_t s, int64_t n, float *w, const float *g, float *m1, float *m2, float lr, float b1, float b2,
               float eps, int step, void *wb) {
  const float c1 = 1.f / (1.f - powf(b1, (float)step)), c2 = 1.f / (1.f - powf(b2, (float)step));
  k_adam<<<1024, 256, 0, s>>>(n, w, g, m1, m2, lr, b1, b2, eps, c1, c2, (__bf16 *)wb);
}

void weights_bf16(hipStream_t s, int64_t n, const float *w, void *wb) {
  k_weights_bf16<<<1024, 256, 0, s>>>(n, w, (__bf16 *)wb);
}

void gather_rows(hipStream_t s, int B, const int *idx, const void *X, const float *T, const unsigned char *rank,
                 void *Xb, float *Tb, unsigned char *rb) {
  k_gather<<<B, 256, 0, s>>>(B, idx, (const __bf16 *)X, T, rank, (__bf16 *)Xb, Tb, rb);
}

}  // namespace ptn
