// MTTKRP building blocks on FP64 matrix cores (v_mfma_f64_16x16x4_f64).
//
// The reference forms M_n = X_(n) * KR explicitly with Eigen GEMM per block
// (MTTKRP.hpp:60-69, :195-220) or streams blocks host->device for cublasDgemm
// (CUDAMTTKRP.hpp:157-175).  Here X stays resident and is read once per
// contraction; Khatri-Rao rows are formed in registers from factor rows; the
// unfolding X_(n) is index arithmetic, never a copy (Matricization.hpp:101-124).
//
// Two GEMM shapes cover every mode of every tree:
//   gemm_cm:  out[m][r] = sum_k X[m + M*k] W(k)[r]   (contracted index strided;
//             mode-0 MTTKRP, the dimension tree's X x_{N-1} A_{N-1})
//   gemm_ck:  T[c][r]   = sum_a X[a + L*c] W(a)[r]   (contracted index contiguous;
//             X x_0 A_0, the dimension tree's right node)
// and contract_rows finishes a contraction against Khatri-Rao rows (the TTVs of
// TensorPartialProduct_R, TensorOperations.hpp:196-213).
//
// MFMA 16x16x4 f64 operand layout (lane l, g = l/16, f = l%16):
//   A (16x4): A[f][g]   B (4x16): B[g][f]   D (16x16): D[g+4v][f], v = 0..3
//   (the D row layout was checked on gfx950 with single-entry tensors)
#include "ptn_internal.hpp"

namespace ptn {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
// 16-byte loads at element alignment (a fibre may start at any element)
typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

namespace {

#include "wave_common.inc"

// The set-up of an NNLS update by one wave, as k_eig_extremes<16> does it.  In a kernel of its own
// it stands in the stream between two contractions and leaves the chip to one block; as one more
// block of the contraction (template parameter SETUP) it is hidden by, or hides, that: sweeps
// of 100^3 at rank 10 205 -> 188 us, 301 x 205 x 150 at 10 257 -> 215, order 4 60 x 50 x 40 x 30 at 8
// 275 -> 246.
__device__ __forceinline__ void nnls_setup_wave(const NnlsSetup &u) {
  __shared__ EigLds<16> S;
  const int l = threadIdx.x & 63;
  for (int x = l; x < 256; x += 64) {
    const int r = x / 16, c = x % 16;
    double v = 0.0;
    if (r < u.R && c < u.R) {
      const int e = r * u.R + c;
      v = u.g[0][e];
      for (int j = 1; j < u.ng; ++j) v = u.g[j][e] * v;
      u.V[e] = v;
    }
    S.t[x] = v;
  }
  PTN_WAVE_SYNC();
  double amax, amin;
  eig_extremes_wave(u.R, S, amax, amin);
  glambda_betas(amax, amin, u.prm, u.max_inner, u.betas);
}

struct KrArgs {
  int nm;
  uint32_t dim[kMaxOrder];
  const double *fac[kMaxOrder];
};

KrArgs to_args(const KrSpec &w) {
  KrArgs a{};
  a.nm = w.nm;
  for (int j = 0; j < w.nm; ++j) { a.dim[j] = (uint32_t)w.dim[j]; a.fac[j] = w.fac[j]; }
  return a;
}

// gemm_cm's loads.  Cached ones: where columns are no whole cache lines, neighbouring ones share
// them, and a non-temporal line is fetched again for each (501 x 403 x 307 at rank 17: 140 us, cached
// 120), and what the 256 MB of the last-level cache hold stays there from one pass to the next.
// NTL: non-temporal ones for FP64 columns of whole lines, and many of them, in a larger tensor, which
// only pass through (left node of 1024^2 x 100 (0.84 GB) at rank 32 260 us cached and 245 so, of 1600 x
// 1248 x 20 (0.32 GB) at 8 211 and 203, mode 0 of 800 x 300 x 300 at 8 113 and 107; but of 128 x 300 x
// 1000 (0.31 GB) at 40 108 and 111, the left node of 4096 x 60 x 60 (118 MB) at 8 34 and 39, and in FP32
// of 640^3 (1 GB) at 8 272 and 293).
template <bool NTL, typename TX>
__device__ __forceinline__ double ld(const TX *p) {
  if constexpr (NTL) return (double)__builtin_nontemporal_load(p);
  else return (double)*p;
}

// ---------------------------------------------------------------------------
// gemm_cm: a block owns 64 consecutive rows and one k-chunk; its 4 waves take
// interleaved k-steps of 4 columns and are summed through LDS at the end.
// ---------------------------------------------------------------------------
template <typename TX, int NT, bool NTL, bool SETUP>
__global__ __launch_bounds__(256, 2) void k_gemm_cm_f64(const TX *__restrict__ X, int64_t Mrows, int64_t Ktot,
                                                     KrArgs w, int ldr, int64_t kchunk, double *__restrict__ out,
                                                     NnlsSetup setup) {
  if constexpr (SETUP) {
    if (blockIdx.x + 1 == gridDim.x) {
      if (blockIdx.y == 0 && threadIdx.x < 64) nnls_setup_wave(setup);
      return;
    }
  }
  constexpr int RP = NT * 16;
  __shared__ double red[64 * RP];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, f = lane & 15;
  const int64_t mb = (int64_t)blockIdx.x * 64;
  const int64_t kbeg = (int64_t)blockIdx.y * kchunk;
  const int64_t kend = kbeg + kchunk < Ktot ? kbeg + kchunk : Ktot;

  f64x4 acc[4][NT];
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[s][t] = f64x4{0.0, 0.0, 0.0, 0.0};

  // Every load is unconditional, so that loads stay in flight across the MFMAs: a row past
  // Mrows reads row Mrows - 1 (its sums are never stored); a column past the chunk reads
  // the chunk's first column and a factor row 0, and both operands of that column are
  // replaced by zero where the MFMAs use them.
  int64_t roff[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int64_t m = mb + 16 * s + f;
    roff[s] = m < Mrows ? m : Mrows - 1;
  }

  // digits of this lane's first column kk = kbeg + 4*wave + g (lowest mode fastest)
  int64_t kk = kbeg + 4 * wave + g;
  uint32_t dig[kMaxOrder];
  {
    uint64_t rem = (uint64_t)kk;
    for (int j = 0; j < w.nm; ++j) { dig[j] = (uint32_t)(rem % w.dim[j]); rem /= w.dim[j]; }
  }
  // The Khatri-Rao values of the lane's current column as two factors, p (the product of
  // all but the last mode's rows, left to right) and q (the last mode's row; 1 for one
  // mode), so that p * q is the left-to-right product and the last multiply can wait
  // until the MFMAs need it; then the odometer advanced by 16.
  auto kr_next = [&](bool kv, double (&p)[NT], double (&q)[NT]) {
    const int last = w.nm - 1;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      double pv = w.fac[0][(int64_t)(kv ? dig[0] : 0u) * ldr + 16 * t + f];
      for (int j = 1; j < last; ++j) pv *= w.fac[j][(int64_t)(kv ? dig[j] : 0u) * ldr + 16 * t + f];
      p[t] = pv;
      q[t] = last > 0 ? w.fac[last][(int64_t)(kv ? dig[last] : 0u) * ldr + 16 * t + f] : 1.0;
    }
    dig[0] += 16;
    for (int j = 0; j + 1 < w.nm && dig[j] >= w.dim[j]; ++j) {
      uint32_t c = dig[j] / w.dim[j];
      dig[j] -= c * w.dim[j];
      dig[j + 1] += c;
    }
  };
  // one step of 16 columns (4 per wave): loads, then (apply) the zeroing and the MFMAs
  auto load_step = [&](bool &kv, double (&a)[4], double (&p)[NT], double (&q)[NT]) {
    kv = kk < kend;
    kr_next(kv, p, q);
    const TX *xp = X + Mrows * (kv ? kk : kbeg);
#pragma unroll
    for (int s = 0; s < 4; ++s) a[s] = ld<NTL>(xp + roff[s]);
    kk += 16;
  };
  auto mma_step = [&](bool kv, const double (&a)[4], const double (&p)[NT], const double (&q)[NT]) {
    double b[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) b[t] = kv ? p[t] * q[t] : 0.0;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const double av = kv ? a[s] : 0.0;
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[s][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, b[t], acc[s][t], 0, 0, 0);
    }
  };
  // Groups of KU steps, software-pipelined over two register buffers: group G+1's loads
  // are issued before group G's MFMAs, with no branch between a load and its use inside
  // the loop.  The MFMAs run in step order (the same sums as one step at a time).
  // (FP32 data at two column tiles: groups of one step, since two steps' converted values
  // overflowed the registers into scratch)
  constexpr int KU = NT == 1 ? 4 : NT == 2 && sizeof(TX) == 8 ? 2 : 1;
  struct Buf {
    bool kv[KU];
    double a[KU][4], p[KU][NT], q[KU][NT];
  };
  auto load_group = [&](Buf &B) {
#pragma unroll
    for (int u = 0; u < KU; ++u) load_step(B.kv[u], B.a[u], B.p[u], B.q[u]);
  };
  auto mma_group = [&](const Buf &B) {
#pragma unroll
    for (int u = 0; u < KU; ++u) mma_step(B.kv[u], B.a[u], B.p[u], B.q[u]);
  };
  const int64_t kw = kk - g;                                 // the wave's first column
  const int64_t nsteps = kend > kw ? (kend - kw + 15) / 16 : 0;
  const int64_t ngroups = nsteps / KU;
  if (ngroups > 0) {
    Buf b0, b1;
    load_group(b0);
    int64_t G = 0;
    for (; G + 2 < ngroups; G += 2) {
      load_group(b1);
      mma_group(b0);
      load_group(b0);
      mma_group(b1);
    }
    if (G + 1 < ngroups) {
      load_group(b1);
      mma_group(b0);
      mma_group(b1);
    } else {
      mma_group(b0);
    }
  }
  for (int64_t j = ngroups * KU; j < nsteps; ++j) {
    bool kv;
    double a[4], p[NT], q[NT];
    load_step(kv, a, p, q);
    mma_step(kv, a, p, q);
  }

  // sum the 4 waves' tiles in LDS, in wave order
  for (int src = 0; src < 4; ++src) {
    if (wave == src) {
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            int row = 16 * s + g + 4 * v, col = 16 * t + f;
            red[row * RP + col] = (src == 0 ? 0.0 : red[row * RP + col]) + acc[s][t][v];
          }
    }
    __syncthreads();
  }
  double *o = out + ((int64_t)blockIdx.y * Mrows) * ldr;
  for (int e = threadIdx.x; e < 64 * RP; e += 256) {
    int row = e / RP, col = e % RP;
    if (mb + row < Mrows) o[(mb + row) * ldr + col] = red[e];
  }
}

// ---------------------------------------------------------------------------
// gemm_ck: a wave (a block of its own) owns 16 S fibers (S MFMA row tiles) and the whole
// contraction.  Within a 16-wide k-block, lane group g supplies a = kb + 4g + t at MFMA
// step t, so each lane reads 4 consecutive elements of its fiber: 32 bytes of FP64 (two
// 16-byte loads) or 16 of FP32 (one), at whatever element the fiber starts.  Reading them
// one by one where the fiber length is not a multiple of 4, and the FP32 tensor always so,
// left the kernel waiting on scattered 8-byte loads with nothing in flight behind them.
// The elements past the last whole block are the end of the block that ends with the fiber
// (wide loads again; the elements that an earlier block had are zeroed): element by element
// under a mask they cost as much as a third of the fiber.
// The loads are cached ones: the two halves of a lane's 32 bytes, and the lines that a block
// of an unaligned fiber shares with the next, are in two loads each, and non-temporal loads
// fetched them twice (800^3 R = 32 node 986 -> 803 us, 5.3 TB/s; 501 x 403 x 307 R = 33, FP64
// tensor 207 -> 156, of 423 at the start; 190 x 155 x 1464 R = 12 127 -> 81).
// S: a Khatri-Rao fragment serves S tiles, so 4 where the fibers fill the chip all the same
// (800^3 R = 32 803 us against 922 at S = 2; 123 721 fibers 156 against 163), 2 below 65 536
// fibers (30 750: 21.4 us against 27.8 at S = 4) and for FP32 tensors, whose conversions take
// the registers of a wave (245 000 fibers 44 against 52 us), 1 below 16 384 (10 000: 5.8 us
// against 6.2 and 7.9).
// ---------------------------------------------------------------------------
template <typename TX, int NT, int S, bool SETUP>
__global__ __launch_bounds__(64, NT * S <= 8 ? 2 : 1) void k_gemm_ck_f64(const TX *__restrict__ X, int64_t L,
                                                                         int64_t C, KrArgs w, int ldr,
                                                                         double *__restrict__ T, NnlsSetup setup) {
  if (SETUP && blockIdx.x == 0) {
    nnls_setup_wave(setup);
    return;
  }
  const int lane = threadIdx.x;
  const int g = lane >> 4, f = lane & 15;
  const int64_t cb = (int64_t)(blockIdx.x - (SETUP ? 1 : 0)) * (16 * S);

  f64x4 acc[S][NT];
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int u = 0; u < NT; ++u) acc[s][u] = f64x4{0.0, 0.0, 0.0, 0.0};

  const TX *xp[S];                              // a fiber past C reads fiber 0; its sums are never stored
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int64_t c = cb + 16 * s + f;
    xp[s] = X + L * (c < C ? c : 0);
  }
  // the Khatri-Rao row of the contracted modes at a (lowest mode fastest), NT fragments
  // (the product runs over the digits as they are split off, so no array of row pointers
  // is indexed at run time: such an array lives in scratch memory)
  auto kr_row = [&](int64_t a, double (&b)[NT]) {
    uint32_t rem = (uint32_t)a;                   // a < L: the last digit is what remains
    for (int j = 0; j < w.nm; ++j) {
      const bool lastd = j + 1 == w.nm;
      const uint32_t d = lastd ? rem : rem % w.dim[j];
      rem = lastd ? 0u : rem / w.dim[j];
      const double *row = w.fac[j] + (int64_t)d * ldr;
#pragma unroll
      for (int u = 0; u < NT; ++u) b[u] = j == 0 ? row[16 * u + f] : b[u] * row[16 * u + f];
    }
  };
  struct Buf {
    TX x[S][4];                                   // (FP32 elements widen where they are multiplied)
    double b[4][NT];
  };
  auto mma16 = [&](const Buf &B) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int u = 0; u < NT; ++u)
          acc[s][u] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)B.x[s][t], B.b[t][u], acc[s][u], 0, 0, 0);
  };
  auto load_blk = [&](int64_t kb, Buf &B) {
#pragma unroll
    for (int t = 0; t < 4; ++t) kr_row(kb + 4 * g + t, B.b[t]);
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if constexpr (sizeof(TX) == 8) {
        const f64x2u *q = (const f64x2u *)(xp[s] + kb + 4 * g);
        const f64x2u lo = q[0], hi = q[1];
        B.x[s][0] = lo[0];
        B.x[s][1] = lo[1];
        B.x[s][2] = hi[0];
        B.x[s][3] = hi[1];
      } else {
        const f32x4u v = *(const f32x4u *)(xp[s] + kb + 4 * g);
#pragma unroll
        for (int j = 0; j < 4; ++j) B.x[s][j] = v[j];
      }
    }
  };
  // zero the block's entries outside [lo, L)
  auto keep_from = [&](int64_t kb, int64_t lo, Buf &B) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int64_t a = kb + 4 * g + t;
      const bool in = a >= lo && a < L;
#pragma unroll
      for (int s = 0; s < S; ++s) B.x[s][t] = in ? B.x[s][t] : (TX)0;
#pragma unroll
      for (int u = 0; u < NT; ++u) B.b[t][u] = in ? B.b[t][u] : 0.0;
    }
  };
  Buf b0, b1;
  if (L >= 16) {
    // Blocks are software-pipelined over two register buffers: block j+1's Khatri-Rao rows
    // and tensor loads are issued before block j's MFMAs, with no branch between a load and
    // its use in the loop.
    const int64_t nblk = (L + 15) / 16, lo = 16 * (nblk - 1);
    auto start = [&](int64_t j) { return 16 * j < L - 16 ? 16 * j : L - 16; };
    load_blk(0, b0);
    int64_t j = 0;
    for (; j + 2 < nblk; j += 2) {
      load_blk(start(j + 1), b1);
      mma16(b0);
      load_blk(start(j + 2), b0);
      mma16(b1);
    }
    if (j + 1 < nblk) {
      load_blk(start(j + 1), b1);
      mma16(b0);
      keep_from(start(j + 1), lo, b1);
      mma16(b1);
    } else {
      keep_from(start(j), lo, b0);
      mma16(b0);
    }
  } else {                                        // a fiber shorter than a block: clamped element loads
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int64_t a = 4 * g + t, ac = a < L ? a : L - 1;
      kr_row(ac, b0.b[t]);
#pragma unroll
      for (int s = 0; s < S; ++s) b0.x[s][t] = __builtin_nontemporal_load(xp[s] + ac);
    }
    keep_from(0, 0, b0);
    mma16(b0);
  }
  // the node leaves with non-temporal stores (a leaf reads it after the other streams' work;
  // 800^3 R = 32 right node 1.020 -> 0.993 ms)
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t c = cb + 16 * s + g + 4 * v;
      if (c < C) {
#pragma unroll
        for (int u = 0; u < NT; ++u) __builtin_nontemporal_store(acc[s][u][v], &T[c * ldr + 16 * u + f]);
      }
    }
}

// ---------------------------------------------------------------------------
// contract_rows: block (i, split) sums, for output index i, the rows of T whose
// remaining digits fall in the split, weighted by the other modes' factor rows.
// Threads: r = tid % RP, group = tid / RP; groups are summed in LDS in order.
//
// A row's digits took two 64-bit divisions each, and the row was waited for before the next
// one's.  With two other modes (order-4 tensors) the digits are carried along from row to row and
// four rows are on their way at once (TWO: 190 x 155 x 61 x 24 at rank 12, mode 2, 23.7 -> 12.1 us).
// ---------------------------------------------------------------------------
struct RowSpec {
  int nm, outmode;
  uint32_t dim[kMaxOrder];
  int64_t stride[kMaxOrder];   // row stride of each digit in T
  const double *fac[kMaxOrder];
};

template <typename TT, bool TWO>
__global__ __launch_bounds__(256) void k_contract_rows(const TT *__restrict__ T, int64_t ldt, RowSpec sp, int RP,
                                                       int ldr, int64_t cchunk, int64_t Cother,
                                                       double *__restrict__ partials, const int *sel,
                                                       int64_t sel_off) {
  if (sel) T += (int64_t)(*sel) * sel_off;              // node chosen on the device (line search)
  __shared__ double red[256];
  const int r = threadIdx.x % RP, grp = threadIdx.x / RP, ngrp = 256 / RP;
  const uint32_t i = blockIdx.x;
  const int64_t c0 = (int64_t)blockIdx.y * cchunk;
  const int64_t c1 = c0 + cchunk < Cother ? c0 + cchunk : Cother;
  double acc = 0.0;
  if constexpr (TWO) {
    const int ja = sp.outmode == 0 ? 1 : 0, jb = sp.outmode == 2 ? 1 : 2;
    const uint32_t Da = sp.dim[ja];
    const int64_t sa = sp.stride[ja] * ldt, sb = sp.stride[jb] * ldt;
    const double *fa = sp.fac[ja] + r, *fb = sp.fac[jb] + r;
    const TT *Ti = T + (int64_t)i * sp.stride[sp.outmode] * ldt + r;
    if (grp < ngrp && c0 + grp < c1) {
      uint32_t da = (uint32_t)((uint64_t)(c0 + grp) % Da), db = (uint32_t)((uint64_t)(c0 + grp) / Da);
      auto advance = [&] {
        da += ngrp;
        while (da >= Da) {
          da -= Da;
          ++db;
        }
      };
      int64_t n = (c1 - c0 - grp + ngrp - 1) / ngrp;    // the thread's rows
      for (; n >= 4; n -= 4) {
        double x[4], wa[4], wb[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          x[u] = (double)Ti[da * sa + db * sb];
          wa[u] = fa[(int64_t)da * ldr];
          wb[u] = fb[(int64_t)db * ldr];
          advance();
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) acc = fma(x[u], wa[u] * wb[u], acc);
      }
      for (; n > 0; --n) {
        acc = fma((double)Ti[da * sa + db * sb], fa[(int64_t)da * ldr] * fb[(int64_t)db * ldr], acc);
        advance();
      }
    }
  } else if (grp < ngrp) {
    for (int64_t c = c0 + grp; c < c1; c += ngrp) {
      uint64_t rem = (uint64_t)c;
      int64_t row = (int64_t)i * sp.stride[sp.outmode];
      double wv = 1.0;
      for (int j = 0; j < sp.nm; ++j) {
        if (j == sp.outmode) continue;
        uint32_t d = (uint32_t)(rem % sp.dim[j]);
        rem /= sp.dim[j];
        row += (int64_t)d * sp.stride[j];
        wv *= sp.fac[j][(int64_t)d * ldr + r];
      }
      acc = fma((double)T[row * ldt + r], wv, acc);
    }
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  if (threadIdx.x < RP) {
    double s = 0.0;
    for (int q = 0; q < ngrp; ++q) s += red[q * RP + threadIdx.x];
    partials[((int64_t)blockIdx.y * gridDim.x + i) * ldr + threadIdx.x] = s;
  }
}

// ---------------------------------------------------------------------------
// contract2: a node with two digits (rows m = i0 + D0 i1, ld values per row) contracted
// over one digit against the other digit's factor rows (a leaf TTV of the dimension
// tree, TensorPartialProduct_R, TensorOperations.hpp:196-213).  Thread (q, c): row
// group q = tid / 32, column c (+ 32 t for the column tiles).  Loads are issued four
// rows at a time; the order of the sums is fixed.
//   outmode 0: block (8 consecutive i0, i1-split), out[i0][r] = sum_i1 Y[m][r] F[i1][r]
//   outmode 1: block (one i1, i0-split), 8 row groups summed in LDS in order
// With gridDim.z == 2 the blocks of z = 1 contract (Y2, F2) beside (Y, F); partials are
// part[split][z][i][ldr].
// ---------------------------------------------------------------------------
template <typename TT>
__global__ __launch_bounds__(256) void k_contract2(const TT *__restrict__ Y, int64_t ld, int64_t D0, int64_t D1,
                                                   int outmode, const double *__restrict__ F, int ldr, int R,
                                                   int64_t slen, double *__restrict__ part, const int *sel,
                                                   int64_t sel_off, const TT *__restrict__ Y2,
                                                   const double *__restrict__ F2) {
  if (sel) Y += (int64_t)(*sel) * sel_off;              // node chosen on the device (line search)
  if (blockIdx.z) {
    Y = Y2;
    F = F2;
  }
  const int64_t zs = (int64_t)blockIdx.y * gridDim.z + blockIdx.z;
  __shared__ double red[8][32];
  const int q = threadIdx.x >> 5, c0 = threadIdx.x & 31;
  const int NT = (R + 31) / 32;
  if (outmode == 0) {
    const int64_t i0 = (int64_t)blockIdx.x * 8 + q;
    const int64_t b = (int64_t)blockIdx.y * slen, e = b + slen < D1 ? b + slen : D1;
    for (int t = 0; t < NT; ++t) {
      const int c = 32 * t + c0;
      if (i0 >= D0 || c >= ldr) continue;
      double acc = 0.0;
      int64_t i1 = b;
      for (; i1 + 4 <= e; i1 += 4) {
        const double y0 = (double)Y[(i0 + D0 * i1) * ld + c], y1 = (double)Y[(i0 + D0 * (i1 + 1)) * ld + c];
        const double y2 = (double)Y[(i0 + D0 * (i1 + 2)) * ld + c], y3 = (double)Y[(i0 + D0 * (i1 + 3)) * ld + c];
        const double f0 = F[i1 * ldr + c], f1 = F[(i1 + 1) * ldr + c];
        const double f2 = F[(i1 + 2) * ldr + c], f3 = F[(i1 + 3) * ldr + c];
        acc = fma(y0, f0, acc);
        acc = fma(y1, f1, acc);
        acc = fma(y2, f2, acc);
        acc = fma(y3, f3, acc);
      }
      for (; i1 < e; ++i1) acc = fma((double)Y[(i0 + D0 * i1) * ld + c], F[i1 * ldr + c], acc);
      part[(zs * D0 + i0) * ldr + c] = acc;
    }
    return;
  }
  const int64_t i1 = blockIdx.x;
  const int64_t b = (int64_t)blockIdx.y * slen, e = b + slen < D0 ? b + slen : D0;
  for (int t = 0; t < NT; ++t) {
    const int c = 32 * t + c0;
    double acc = 0.0;
    if (c < ldr) {
      const TT *row = Y + (D0 * i1) * ld + c;
      int64_t i0 = b + q;
      for (; i0 + 24 < e; i0 += 32) {
        const double y0 = (double)row[i0 * ld], y1 = (double)row[(i0 + 8) * ld];
        const double y2 = (double)row[(i0 + 16) * ld], y3 = (double)row[(i0 + 24) * ld];
        const double f0 = F[i0 * ldr + c], f1 = F[(i0 + 8) * ldr + c];
        const double f2 = F[(i0 + 16) * ldr + c], f3 = F[(i0 + 24) * ldr + c];
        acc = fma(y0, f0, acc);
        acc = fma(y1, f1, acc);
        acc = fma(y2, f2, acc);
        acc = fma(y3, f3, acc);
      }
      for (; i0 < e; i0 += 8) acc = fma((double)row[i0 * ld], F[i0 * ldr + c], acc);
    }
    __syncthreads();
    red[q][c0] = acc;
    __syncthreads();
    if (q == 0 && c < ldr) {
      double sum = red[0][c0];
      for (int g = 1; g < 8; ++g) sum += red[g][c0];
      part[(zs * D1 + i1) * ldr + c] = sum;
    }
  }
}

// k_contract2's outmode 0 for FP32 nodes with 16-byte loads: thread (rr = tid / 8, c4 = tid % 8)
// owns row i0 = 32 bx + rr and columns 4 c4 .. 4 c4 + 3 of each 32-column group; each column
// sums its i1 range in the same order as k_contract2, so the partials are bitwise equal.
// Rows of Y hold ld floats, ld and the node's offset multiples of 4 (16-byte aligned).
__global__ __launch_bounds__(256) void k_contract2_r4(const float *__restrict__ Y, int64_t ld, int64_t D0, int64_t D1,
                                                      const double *__restrict__ F, int ldr, int64_t slen,
                                                      double *__restrict__ part, const int *sel, int64_t sel_off,
                                                      const float *__restrict__ Y2, const double *__restrict__ F2) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  if (sel) Y += (int64_t)(*sel) * sel_off;
  if (blockIdx.z) {
    Y = Y2;
    F = F2;
  }
  const int64_t zs = (int64_t)blockIdx.y * gridDim.z + blockIdx.z;
  const int rr = threadIdx.x >> 3, c4 = 4 * (threadIdx.x & 7);
  const int64_t i0 = (int64_t)blockIdx.x * 32 + rr;
  if (i0 >= D0) return;
  const int64_t b = (int64_t)blockIdx.y * slen, e = b + slen < D1 ? b + slen : D1;
  for (int cb = 0; cb < ldr; cb += 32) {
    const int c = cb + c4;
    if (c >= ldr) break;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    int64_t i1 = b;
    for (; i1 + 4 <= e; i1 += 4) {
      f4 y[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) y[u] = *(const f4 *)(Y + (i0 + D0 * (i1 + u)) * ld + c);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double *f = F + (i1 + u) * ldr + c;
        a0 = fma((double)y[u][0], f[0], a0);
        a1 = fma((double)y[u][1], f[1], a1);
        a2 = fma((double)y[u][2], f[2], a2);
        a3 = fma((double)y[u][3], f[3], a3);
      }
    }
    for (; i1 < e; ++i1) {
      const f4 y = *(const f4 *)(Y + (i0 + D0 * i1) * ld + c);
      const double *f = F + i1 * ldr + c;
      a0 = fma((double)y[0], f[0], a0);
      a1 = fma((double)y[1], f[1], a1);
      a2 = fma((double)y[2], f[2], a2);
      a3 = fma((double)y[3], f[3], a3);
    }
    double *o = part + (zs * D0 + i0) * ldr + c;
    o[0] = a0;
    o[1] = a1;
    o[2] = a2;
    o[3] = a3;
  }
}

// A small FP64 node contracted over one digit, a block to an output row: the columns' threads in
// 256 / ldr groups, each taking every so many-th row with four in flight, the groups summed in LDS in
// order.  k_contract2 splits such a node to fill the chip and has the splits summed by another
// launch, 2 to 5 us of the 6 to 20 that both take (MTTKRP of 200^3 at rank 16 68 -> 64 us, the rule for
// it in contract_node).
__global__ __launch_bounds__(256) void k_contract2_rows(const double *__restrict__ Y, int64_t rstride, int64_t ostride,
                                                        int n, const double *__restrict__ F, int ldr,
                                                        double *__restrict__ out) {
  __shared__ double red[256];
  const int r = threadIdx.x % ldr, g = threadIdx.x / ldr, G = 256 / ldr;
  const double *y = Y + blockIdx.x * ostride + r, *f = F + r;
  double acc = 0.0;
  if (g < G) {
    int j = g;
    for (; j + 3 * G < n; j += 4 * G) {
      double x[4], w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        x[u] = y[(j + u * G) * rstride];
        w[u] = f[(int64_t)(j + u * G) * ldr];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) acc = fma(x[u], w[u], acc);
    }
    for (; j < n; j += G) acc = fma(y[j * rstride], f[(int64_t)j * ldr], acc);
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  if ((int)threadIdx.x < ldr) {
    double s = red[threadIdx.x];
    for (int q = 1; q < G; ++q) s += red[q * ldr + threadIdx.x];
    out[(int64_t)blockIdx.x * ldr + threadIdx.x] = s;
  }
}

__global__ void k_reduce_splits(const double *__restrict__ partials, int splits, int64_t n, double *__restrict__ out) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    double s = 0.0;
    for (int q = 0; q < splits; ++q) s += partials[q * n + e];
    out[e] = s;
  }
}
// the same sums two at a time (n % 2 == 0): 16-byte loads of every split, in split order
__global__ void k_reduce_splits_x2(const f64x2 *__restrict__ partials, int splits, int64_t n2,
                                   f64x2 *__restrict__ out) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n2; e += (int64_t)gridDim.x * blockDim.x) {
    f64x2 s = {0.0, 0.0};
    int q = 0;
    for (; q + 8 <= splits; q += 8) {           // eight loads in flight (39 splits of 100 rows 11 -> 6 us)
      f64x2 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = partials[(q + j) * n2 + e];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        s[0] += v[j][0];
        s[1] += v[j][1];
      }
    }
    for (; q < splits; ++q) {
      const f64x2 v = partials[q * n2 + e];
      s[0] += v[0];
      s[1] += v[1];
    }
    out[e] = s;
  }
}

// Many splits, two sums at a time: eight threads share a sum, each adds a run of splits in order
// with eight loads in flight and the eight meet in LDS, in order.  One thread to a sum is a chain of
// round trips to memory that nothing hides, and a small result has few such threads: the
// FP64 MTTKRP of mode 0 with its 39 splits at 100^3, rank 10 17.3 -> 14.4 us, 200^3 at 32 41 -> 34.6.
__global__ __launch_bounds__(256) void k_reduce_splits_runs(const f64x2 *__restrict__ partials, int splits, int64_t n2,
                                                            f64x2 *__restrict__ out) {
  __shared__ f64x2 run[8][32];
  const int q = threadIdx.x >> 5, l = threadIdx.x & 31;
  const int64_t e = (int64_t)blockIdx.x * 32 + l;
  const int b = q * splits / 8, end = (q + 1) * splits / 8;
  f64x2 s = {0.0, 0.0};
  if (e < n2)
    for (int p = b; p < end; p += 8) {
      f64x2 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = partials[(p + j < end ? p + j : p) * n2 + e];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (p + j < end) {
          s[0] += v[j][0];
          s[1] += v[j][1];
        }
    }
  run[q][l] = s;
  __syncthreads();
  if (q == 0 && e < n2) {
    f64x2 t = run[0][l];
#pragma unroll
    for (int j = 1; j < 8; ++j) {
      t[0] += run[j][l][0];
      t[1] += run[j][l][1];
    }
    out[e] = t;
  }
}

}  // namespace

bool gemm_cm_f64(hipStream_t s, const double *x64, const float *x32, int64_t Mrows, int64_t Ktot, const KrSpec &w,
                 int ldr, int splits, double *out, const NnlsSetup *setup) {
  KrArgs a = to_args(w);
  int64_t kchunk = (Ktot + splits - 1) / splits;
  dim3 grid((unsigned)((Mrows + 63) / 64), (unsigned)splits);
  const int NT = ldr / 16;
  const bool ntl = x64 && Mrows % 16 == 0 && Mrows >= 512 && Mrows * Ktot > ((int64_t)32 << 20);   // (ld)
  if (setup && NT == 1) grid.x += 1;               // one more block
#define PTN_CML(TXV, PTR, NTV, NTLV, SETUPV, UP) \
  k_gemm_cm_f64<TXV, NTV, NTLV, SETUPV><<<grid, 256, 0, s>>>(PTR, Mrows, Ktot, a, ldr, kchunk, out, UP)
#define PTN_CMK(NTV, SETUPV, UP)                              \
  do {                                                        \
    if (ntl) PTN_CML(double, x64, NTV, true, SETUPV, UP);       \
    else if (x64) PTN_CML(double, x64, NTV, false, SETUPV, UP); \
    else PTN_CML(float, x32, NTV, false, SETUPV, UP);           \
  } while (0)
  if (setup && NT == 1) {
    PTN_CMK(1, true, *setup);
    return true;
  }
  const NnlsSetup none{};
#define PTN_CM(NTV)              \
  if (NT == NTV) {               \
    PTN_CMK(NTV, false, none);   \
    return false;                \
  }
  PTN_CM(1) PTN_CM(2) PTN_CM(3) PTN_CM(4)
#undef PTN_CM
#undef PTN_CMK
#undef PTN_CML
  return false;
}

bool gemm_ck_f64(hipStream_t s, const double *x64, const float *x32, int64_t L, int64_t C, const KrSpec &w, int ldr,
                 double *T, const NnlsSetup *setup) {
  KrArgs a = to_args(w);
  const int NT = ldr / 16;
  if (NT != 1) setup = nullptr;
  // Fibers per wave: many share each Khatri-Rao fragment, few leave more waves for the 1024
  // SIMDs (k_gemm_ck_f64)
  const int S = C >= 65536 && x64 ? 4 : C >= 16384 ? 2 : 1;
  const unsigned grid = (unsigned)((C + 16 * S - 1) / (16 * S)) + (setup ? 1 : 0);
  const NnlsSetup none{};
#define PTN_CKS(NTV, SV, UV)                                                                              \
  if (x64) k_gemm_ck_f64<double, NTV, SV, UV><<<grid, 64, 0, s>>>(x64, L, C, a, ldr, T, UV ? *setup : none); \
  else     k_gemm_ck_f64<float, NTV, SV, UV><<<grid, 64, 0, s>>>(x32, L, C, a, ldr, T, UV ? *setup : none);
#define PTN_CK(NTV, UV)              \
  if (NT == NTV) {               \
    if (S == 4) { PTN_CKS(NTV, 4, UV) } \
    else if (S == 2) { PTN_CKS(NTV, 2, UV) } \
    else { PTN_CKS(NTV, 1, UV) }     \
    return setup != nullptr;     \
  }
  if (setup) { PTN_CK(1, true) }
  PTN_CK(1, false) PTN_CK(2, false) PTN_CK(3, false) PTN_CK(4, false)
#undef PTN_CK
#undef PTN_CKS
  return false;
}

void contract_rows(hipStream_t s, const double *T64, const float *T32, int64_t ldt, const KrSpec &spec, int outmode,
                   int ldr, int splits, double *partials, const int *sel, int64_t sel_off) {
  RowSpec sp{};
  sp.nm = spec.nm;
  sp.outmode = outmode;
  int64_t st = 1, Cother = 1;
  for (int j = 0; j < spec.nm; ++j) {
    sp.dim[j] = (uint32_t)spec.dim[j];
    sp.stride[j] = st;
    st *= spec.dim[j];
    sp.fac[j] = spec.fac[j];
    if (j != outmode) Cother *= spec.dim[j];
  }
  int RP = ldr;
  int64_t cchunk = (Cother + splits - 1) / splits;
  dim3 grid((unsigned)spec.dim[outmode], (unsigned)splits);
#define PTN_CR(TTV, PTR)                                                                                        \
  do {                                                                                                          \
    if (spec.nm == 3)                                                                                           \
      k_contract_rows<TTV, true><<<grid, 256, 0, s>>>(PTR, ldt, sp, RP, ldr, cchunk, Cother, partials, sel, sel_off); \
    else                                                                                                        \
      k_contract_rows<TTV, false><<<grid, 256, 0, s>>>(PTR, ldt, sp, RP, ldr, cchunk, Cother, partials, sel, sel_off); \
  } while (0)
  if (T64) PTN_CR(double, T64);
  else PTN_CR(float, T32);
#undef PTN_CR
}

void contract2(hipStream_t s, const double *Y64, const float *Y32, int64_t ld, int64_t D0, int64_t D1, int outmode,
               const double *F, int ldr, int R, int splits, double *part, const int *sel, int64_t sel_off) {
  const int64_t D = outmode == 0 ? D1 : D0;             // contracted extent
  const int64_t slen = (D + splits - 1) / splits;
  dim3 grid(outmode == 0 ? (unsigned)((D0 + 7) / 8) : (unsigned)D1, (unsigned)splits);
  if (Y64)
    k_contract2<double><<<grid, 256, 0, s>>>(Y64, ld, D0, D1, outmode, F, ldr, R, slen, part, sel, sel_off, nullptr,
                                             nullptr);
  else if (outmode == 0 && ld % 4 == 0 && sel_off % 4 == 0 && ((uintptr_t)Y32 & 15) == 0)
    k_contract2_r4<<<dim3((unsigned)((D0 + 31) / 32), (unsigned)splits), 256, 0, s>>>(
        Y32, ld, D0, D1, F, ldr, slen, part, sel, sel_off, nullptr, nullptr);
  else
    k_contract2<float><<<grid, 256, 0, s>>>(Y32, ld, D0, D1, outmode, F, ldr, R, slen, part, sel, sel_off, nullptr,
                                            nullptr);
}

void contract2_rows(hipStream_t s, const double *Y, int64_t ld, int64_t D0, int64_t D1, int outmode, const double *F,
                    int ldr, double *out) {
  if (outmode == 0) k_contract2_rows<<<(unsigned)D0, 256, 0, s>>>(Y, D0 * ld, ld, (int)D1, F, ldr, out);
  else k_contract2_rows<<<(unsigned)D1, 256, 0, s>>>(Y, ld, D0 * ld, (int)D0, F, ldr, out);
}

void contract2_pair(hipStream_t s, const float *Ya, const float *Yb, int64_t ld, int64_t D0, int64_t D1, int outmode,
                    const double *Fa, const double *Fb, int ldr, int R, int splits, double *part) {
  const int64_t D = outmode == 0 ? D1 : D0;
  const int64_t slen = (D + splits - 1) / splits;
  if (outmode == 0 && ld % 4 == 0 && ((uintptr_t)Ya & 15) == 0 && ((uintptr_t)Yb & 15) == 0) {
    k_contract2_r4<<<dim3((unsigned)((D0 + 31) / 32), (unsigned)splits, 2), 256, 0, s>>>(
        Ya, ld, D0, D1, Fa, ldr, slen, part, nullptr, 0, Yb, Fb);
    return;
  }
  dim3 grid(outmode == 0 ? (unsigned)((D0 + 7) / 8) : (unsigned)D1, (unsigned)splits, 2);
  k_contract2<float><<<grid, 256, 0, s>>>(Ya, ld, D0, D1, outmode, Fa, ldr, R, slen, part, nullptr, 0, Yb, Fb);
}

void reduce_splits(hipStream_t s, const double *partials, int splits, int64_t n, double *out, bool runs) {
  if (n % 2 == 0 && ((uintptr_t)partials | (uintptr_t)out) % 16 == 0) {
    if (runs && splits >= 16) {
      k_reduce_splits_runs<<<(unsigned)((n / 2 + 31) / 32), 256, 0, s>>>((const f64x2 *)partials, splits, n / 2,
                                                                         (f64x2 *)out);
      return;
    }
    int64_t g = (n / 2 + 255) / 256;
    if (g > 8192) g = 8192;
    k_reduce_splits_x2<<<(unsigned)g, 256, 0, s>>>((const f64x2 *)partials, splits, n / 2, (f64x2 *)out);
    return;
  }
  int64_t g = (n + 255) / 256;
  if (g > 4096) g = 4096;
  k_reduce_splits<<<(unsigned)g, 256, 0, s>>>(partials, splits, n, out);
}

}  // namespace ptn
