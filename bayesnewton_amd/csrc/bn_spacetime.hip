// Space-time Markov GP (SpatioTemporalKernel, bayesnewton/kernels.py:385-586, with the
// model path of basemodels.py:667-764) on gfx950: K independent runs, each a
// sequence of T steps with R observation locations and M spatial inducing points.
//
// State layout: x = [c = 0 block: f_0..f_{M-1} | c = 1 block: f'_0..f'_{M-1} | ...],
// state index c*M + m, D = KT*M (KT = temporal state dim).  H picks the c = 0 block,
// A = A_t (x) I_M and Q = Q_t (x) I_M act on (c, c') pairs of M x M blocks.
//
// Kernels (all FP64):
//   k_st_conditional  block per (step, run): B_t = Krz Lzz^-T rows, diag C_t     (kernels.py:486-506)
//   k_st_sites        block per (step, run): posterior -> data (basemodels.py:743-764), site
//                     update (inference.py:65-90, 105-195) or energy terms, and the projected
//                     pseudo observation in whitened form: W = B' diag(nat2) B + 1e-12 I = L L',
//                     z = L^-1 B' nat1 (basemodels.py:676-687 without forming W^-1), on register
//                     tiles.  k_st_sites_ordered: the same with every sum in one fixed order,
//                     for the mean-field filter and the EP update, whose results multiply a
//                     last place of L L' by its condition.
//   k_st_transitions  A_t, Q_t of every step.
//   k_st_filter       block per run, loop over T: predict, measurement update in whitened form
//                     with Mm = I + L' Sh L = Lm Lm', W = U Lm^-T, P = P- - W W'.
//                     Equal to ops.py:159-171 with noise (W + 1e-12 I)^-1.
//   k_st_ell          log likelihood terms of every step from what the filter leaves.
//   k_st_gains        block per (step, run): the RTS map of a step (ops.py:288-311) as an affine
//                     map of the next smoothed moments, by a blocked Cholesky of P-.
//   k_st_smoother     the maps applied from the last step back: a walk over all steps of a run,
//                     or, for few runs, chunks of steps composed, joined and walked side by side
//                     (k_st_chain, k_st_terminal: the chunks' ends).
//                     An adjoint (Bryson-Frazier) backward pass avoids the factorisation but
//                     its covariance error grows geometrically over long runs with
//                     precise sites, so the filtered moments are stored instead.
//   k_st_sum          per-run FP64 sums of per-step partials.
//   k_ih_*            the infinite-horizon forms (ops.py:796-1068): per-run Riccati iterations
//                     for a steady-state covariance and gain, means only over the data.
//   k_mf_*            the mean-field forms of the filter and smoother (block-diagonal state
//                     covariance, ops.py:429-706): per-run sequential filter with one M x M
//                     inverse per step, the associative form as per-step M x M work plus a
//                     scalar filter per (run, block) lane, and a per-lane RTS smoother.
// Dense products are FP64 matrix instructions on 16 x 16 tiles held in registers (bn_tile.h), in
// the remaining kernels workgroup GEMMs on operands staged through LDS.
#include <hip/hip_runtime.h>

#include <cmath>
#include <string>

#include "bn_core.h"
#include "bn_internal.h"
#include "bn_sites.h"
#include "bn_tile.h"

using namespace bn;

namespace {

constexpr int kT = 256;      // threads per workgroup
constexpr int kMaxM = 64;    // inducing points per run
constexpr int kMaxKT = 2;    // temporal state dim (Matern12 / Matern32)
constexpr int kMaxD = kMaxKT * kMaxM;  // state dim
constexpr int kPK = 16;      // GEMM K-panel
constexpr int kPS = 68;      // LDS panel row stride (doubles)
constexpr double kPseudoJitter = 1e-12;  // basemodels.py:683

int st_fail(int code, const std::string& msg) { return set_error(code, msg); }

#define ST_HIP_CHECK(expr)                                                                  \
  do {                                                                                      \
    hipError_t e_ = (expr);                                                                 \
    if (e_ != hipSuccess) return st_fail(BN_EHIP, std::string(#expr ": ") + hipGetErrorString(e_)); \
  } while (0)

// element (i, j) of a strided matrix view
struct MatRef {
  const double* p;
  int64_t rs, cs;
  __device__ double at(int i, int j) const { return p[i * rs + j * cs]; }
};

typedef double f64x4 __attribute__((ext_vector_type(4)));

// C[i*ldc + j] = alpha * sum_k A(i,k) B(k,j) + beta * C[i*ldc + j], 0 <= i < m, 0 <= j < n.
// The whole workgroup (kT threads = 4 waves) calls it; every 64x64 output block is
// computed by FP64 matrix-core instructions, one 32x32 quadrant per wave.  Panels of A
// and B go through LDS (`sm`: 2 * kPK * kPS doubles); the next panel is fetched from
// memory into registers while the current one is multiplied.
// Operands and C may live in global memory or LDS; C must not alias A or B.
__device__ void wg_gemm_small(int m, int n, int k, double alpha, MatRef A, MatRef B, double beta, double* C,
                              int64_t ldc, double* sm) {
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  __syncthreads();  // the caller's writes to the operands are complete
  double* As = sm;             // [kPK][kPS]: As[kk][ii] = A(i0+ii, k0+kk)
  double* Bs = sm + kPK * kPS;  // [kPK][kPS]: Bs[kk][jj] = B(k0+kk, j0+jj)
  constexpr int NL = kPK * 64 / kT;  // panel elements loaded per thread
  for (int i0 = 0; i0 < m; i0 += 64) {
    for (int j0 = 0; j0 < n; j0 += 64) {
      f64x4 acc[2][2];
#pragma unroll
      for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj) acc[bi][bj] = f64x4{0.0, 0.0, 0.0, 0.0};
      // the next panel is fetched into registers while the current one is used
      double ra[NL], rb[NL];
      auto fetch = [&](int k0) {
#pragma unroll
        for (int q = 0; q < NL; ++q) {
          const int e = tid + q * kT;
          int ii, kk, jj, kk2;
          if (A.cs == 1) { ii = e >> 4; kk = e & 15; } else { kk = e >> 6; ii = e & 63; }
          if (B.cs == 1) { kk2 = e >> 6; jj = e & 63; } else { jj = e >> 4; kk2 = e & 15; }
          const int gi = i0 + ii, gk = k0 + kk, gj = j0 + jj, gk2 = k0 + kk2;
          ra[q] = (gi < m && gk < k) ? A.at(gi, gk) : 0.0;
          rb[q] = (gj < n && gk2 < k) ? B.at(gk2, gj) : 0.0;
        }
      };
      fetch(0);
      for (int k0 = 0; k0 < k; k0 += kPK) {
#pragma unroll
        for (int q = 0; q < NL; ++q) {
          const int e = tid + q * kT;
          int ii, kk, jj, kk2;
          if (A.cs == 1) { ii = e >> 4; kk = e & 15; } else { kk = e >> 6; ii = e & 63; }
          if (B.cs == 1) { kk2 = e >> 6; jj = e & 63; } else { jj = e >> 4; kk2 = e & 15; }
          As[kk * kPS + ii] = ra[q];
          Bs[kk2 * kPS + jj] = rb[q];
        }
        __syncthreads();
        if (k0 + kPK < k) fetch(k0 + kPK);
        // wave w: 32 x 32 quadrant (rows (w/2)*32, cols (w%2)*32) as 2 x 2 blocks of
        // v_mfma_f64_16x16x4f64: lane l holds A[l%16][k+l/16], B[k+l/16][l%16]
#pragma unroll
        for (int kk = 0; kk < kPK; kk += 4) {
          double af[2], bf[2];
#pragma unroll
          for (int bi = 0; bi < 2; ++bi) af[bi] = As[(kk + (lane >> 4)) * kPS + wr + bi * 16 + (lane & 15)];
#pragma unroll
          for (int bj = 0; bj < 2; ++bj) bf[bj] = Bs[(kk + (lane >> 4)) * kPS + wc + bj * 16 + (lane & 15)];
#pragma unroll
          for (int bi = 0; bi < 2; ++bi)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj) acc[bi][bj] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[bi], bf[bj], acc[bi][bj], 0, 0, 0);
        }
        __syncthreads();
      }
      // output: block (bi, bj), register r -> row wr + bi*16 + lane/16 + 4r, column wc + bj*16 + lane%16
#pragma unroll
      for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int gi = i0 + wr + bi * 16 + (lane >> 4) + 4 * r;
            const int gj = j0 + wc + bj * 16 + (lane & 15);
            if (gi < m && gj < n) {
              double v = alpha * acc[bi][bj][r];
              if (beta != 0.0) v = fma(beta, C[gi * ldc + gj], v);
              C[gi * ldc + gj] = v;
            }
          }
    }
  }
  __syncthreads();
}

// In-place inverse of an n x n symmetric positive definite matrix a (LDS, stride ld) by
// the sweep operator on every pivot: a := -a^-1.  Returns sum log pivots = log det a
// (thread 0 only, when LOGDET).  Diagonal pivots of an SPD matrix stay positive, so no pivoting;
// a non-positive pivot gives NaN, which propagates.  Thread t holds, in registers, the
// B x B elements at rows t/16 + 16 i and columns t%16 + 16 j (cyclic, n <= 16 B): pivot
// k = 16 ib + rr then sits in register row/column ib for every thread, a compile-time
// index once ib is unrolled, so the pivot row and column fix-ups are predicated selects.
// Per pivot the owners of row k publish it to LDS (`row`: 2 x 16B doubles,
// double-buffered); by symmetry it is also column k.
template <int B, bool LOGDET>
__device__ double wg_sweep_inv(double* a, int n, int ld, double* row) {
  const int tid = threadIdx.x;
  const int rg = tid >> 4, cg = tid & 15;
  double v[B][B];
  __syncthreads();  // the caller's writes to `a` are complete
#pragma unroll
  for (int i = 0; i < B; ++i)
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const int gi = rg + 16 * i, gj = cg + 16 * j;
      v[i][j] = (gi < n && gj < n) ? a[gi * ld + gj] : 0.0;
    }
  double logdet = 0.0;
  __syncthreads();
#pragma unroll
  for (int ib = 0; ib < B; ++ib) {
    const int kend = min(16, n - 16 * ib);
    for (int rr = 0; rr < kend; ++rr) {
      const int k = 16 * ib + rr;
      double* rw = row + (k & 1) * (16 * B);
      if (rg == rr) {
#pragma unroll
        for (int j = 0; j < B; ++j) rw[cg + 16 * j] = v[ib][j];
      }
      __syncthreads();
      const double d = rw[k];
      const double id = 1.0 / d;
      if (LOGDET && tid == 0) logdet += log(d);
      double ri[B], rj[B];
#pragma unroll
      for (int i = 0; i < B; ++i) { ri[i] = rw[rg + 16 * i] * id; rj[i] = rw[cg + 16 * i]; }
      // generic rank-1 update, then the pivot row / column of the owners:
      // a_kj := a_kj / d, a_ik := a_ik / d, a_kk := -1 / d
#pragma unroll
      for (int i = 0; i < B; ++i)
#pragma unroll
        for (int j = 0; j < B; ++j) v[i][j] = fma(-ri[i], rj[j], v[i][j]);
      const bool orow = rg == rr, ocol = cg == rr;
#pragma unroll
      for (int j = 0; j < B; ++j) v[ib][j] = orow ? rj[j] * id : v[ib][j];
#pragma unroll
      for (int i = 0; i < B; ++i) v[i][ib] = ocol ? ((i == ib && orow) ? -id : ri[i]) : v[i][ib];
    }
  }
#pragma unroll
  for (int i = 0; i < B; ++i)
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const int gi = rg + 16 * i, gj = cg + 16 * j;
      if (gi < n && gj < n) a[gi * ld + gj] = v[i][j];
    }
  __syncthreads();
  return logdet;
}

// Forward substitution L X = B for `nrhs` right-hand-side columns, one thread per
// column (L lower n x n in LDS with stride ld; B(i, c) = b[i*bs + c*bcs], solved in place).
__device__ void wg_lower_solve(const double* L, int n, int ld, double* b, int bs, int bcs, int nrhs) {
  const int tid = threadIdx.x;
  __syncthreads();
  for (int c = tid; c < nrhs; c += kT) {
    double* x = b + c * bcs;
    for (int i = 0; i < n; ++i) {
      double s = x[i * bs];
      for (int q = 0; q < i; ++q) s = fma(-L[i * ld + q], x[q * bs], s);
      x[i * bs] = s / L[i * ld + i];
    }
  }
  __syncthreads();
}

// Block sum of one double per thread; result valid in every thread.
__device__ double wg_sum(double v, double* red) {
  const int tid = threadIdx.x;
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();
  if ((tid & 63) == 0) red[tid >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int w = 0; w < kT / 64; ++w) s += red[w];
  __syncthreads();
  return s;
}

struct StDims {
  int32_t K, T, R, M, KT, D;
};

// Temporal hypers (one set per run, stride 0 shares one set) and spatial variance.
struct StHyp {
  const double* ls_t;
  const double* var_t;
  const double* var_s;
  int32_t stride;
};

template <int KT>
__device__ void temporal_AQ(double ls, double var, double dt, double A[KT * KT], double Q[KT * KT]) {
  Model<KT, 0> mdl;
  mdl.init(ls, var, 1.0, 1.0);
  double Am[KT][KT], Qm[KT][KT];
  mdl.discretise(dt, Am, Qm);
  for (int i = 0; i < KT; ++i)
    for (int j = 0; j < KT; ++j) { A[i * KT + j] = Am[i][j]; Q[i * KT + j] = Qm[i][j]; }
}

// Matern correlation at scaled distance r (kernels.py:130-133, 182-186, 240-245).
__device__ inline double spatial_corr(int32_t kind, double r) {
  if (kind == BN_MATERN12) return exp(-r);
  if (kind == BN_MATERN32) {
    const double a = sqrt(3.0) * r;
    return (1.0 + a) * exp(-a);
  }
  const double a = sqrt(5.0) * r;
  return (1.0 + a + 5.0 / 3.0 * r * r) * exp(-a);
}

// ---------------------------------------------------------------------------
// k_st_conditional: B_t rows (b_i = Lzz^-1 k(z, r_i)) and diag C_t = var_t (var_s - |b_i|^2)
// kernels.py:486-506 (K = Krz Kzz^-1, B = K Lzz = Krz Lzz^-T; C = k_t(0)(Krr - K Krz')).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kT) void k_st_conditional(StDims dm, StHyp hy, const double* __restrict__ Lzz,
                                                       const double* __restrict__ z, int32_t skind, double ls_s,
                                                       const float* __restrict__ r, double* __restrict__ B,
                                                       double* __restrict__ cdiag) {
  __shared__ double sL[kMaxM * kMaxM];
  __shared__ double sz[kMaxM * 2];
  const int t = blockIdx.x, k = blockIdx.y, M = dm.M;
  const int tid = threadIdx.x;
  for (int e = tid; e < M * M; e += kT) sL[e] = Lzz[e];
  for (int e = tid; e < 2 * M; e += kT) sz[e] = z[e];
  __syncthreads();
  const double vt = hy.var_t[k * hy.stride], vs = hy.var_s[k * hy.stride];
  const double il = 1.0 / ls_s;
  const int64_t base = ((int64_t)k * dm.T + t) * dm.R;
  for (int i = tid; i < dm.R; i += kT) {
    const double rx = r[(base + i) * 2], ry = r[(base + i) * 2 + 1];
    double b[kMaxM];
    double nb = 0.0;
    for (int j = 0; j < M; ++j) {
      const double dx = rx - sz[2 * j], dy = ry - sz[2 * j + 1];
      const double r1 = sqrt(fmax((dx * dx + dy * dy) * il * il, 1e-36));   // kernels.py:101-104
      double s = vs * spatial_corr(skind, r1);
      for (int q = 0; q < j; ++q) s = fma(-sL[j * M + q], b[q], s);
      b[j] = s / sL[j * M + j];
      nb = fma(b[j], b[j], nb);
    }
    double* Bi = B + (base + i) * M;
    for (int j = 0; j < M; ++j) Bi[j] = b[j];
    cdiag[base + i] = vt * (vs - nb);
  }
}

// ---------------------------------------------------------------------------
// k_st_sites: per (step, run).
//   mean_f = B m, var_f = diag(B P B') + diag C  (basemodels.py:743-764)
//   UPDATE: site step of METHOD at (mean_f, var_f), damping with lr, then the whitened
//           pseudo observation L L' = B' diag(nat2) B + 1e-12 I, z = L^-1 B' nat1,
//           ldl = sum log diag L.  part[0] = sum |dnat1|, part[1] = sum |dnat2|.
//   PROJECT: only the whitened pseudo observation of the current sites.
//   ENERGY: part[0] = sum of site terms t1 (inference.py:130-222),
//           part[1] = E_q[log N(pseudo_y | f, pseudo_var)] in whitened form
//           (utils.py:510-531): -1/2(|z - L'm|^2 + M log 2pi - 2 ldl) - 1/2 tr(L' P L).
// ---------------------------------------------------------------------------
struct StSiteIO {
  const float* y;         // [K,T,R]
  const double* B;        // [K,T,R,M]
  const double* cdiag;    // [K,T,R]
  const double* pm;       // [K,T,M]
  const double* pP;       // [K,T,M,M]
  double* nat1;           // [K,T,R]
  double* nat2;           // [K,T,R]
  double* Lw;             // [K,T,M,M]
  double* zw;             // [K,T,M]
  double* ldl;            // [K,T]
  double* part0;          // [K,T]
  double* part1;          // [K,T]
  float* o_mean;          // optional [K,T,R] returned site terms
  float* o_jac;
  float* o_hess;
  const float* batch;     // optional [K,T]: nonzero = step in the mini-batch (NULL: every step)
};

// In-place lower Cholesky of an n x n SPD matrix a (LDS, stride ld), the upper part
// zeroed; register blocks as in wg_sweep_inv, one barrier per pivot.  Returns
// sum log diag L (thread 0 only).  A non-positive pivot gives NaN.
template <int B>
__device__ double wg_chol_reg(double* a, int n, int ld, double* row) {
  const int tid = threadIdx.x;
  const int r0 = (tid >> 4) * B, c0 = (tid & 15) * B;
  double v[B][B];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < B; ++i)
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const int gi = r0 + i, gj = c0 + j;
      v[i][j] = (gi < n && gj < n) ? a[gi * ld + gj] : 0.0;
    }
  double ldl = 0.0;
  for (int k = 0; k < n; ++k) {
    double* rw = row + (k & 1) * (16 * B);
    if (k >= r0 && k < r0 + B) {
#pragma unroll
      for (int i = 0; i < B; ++i)
        if (r0 + i == k) {
#pragma unroll
          for (int j = 0; j < B; ++j) rw[c0 + j] = v[i][j];
        }
    }
    __syncthreads();
    const double d = sqrt(rw[k]);
    const double id = 1.0 / d;
    if (tid == 0) ldl += log(d);
    double ri[B], rj[B];
#pragma unroll
    for (int i = 0; i < B; ++i) {
      ri[i] = (r0 + i > k) ? rw[r0 + i] * id : 0.0;
      rj[i] = (c0 + i > k) ? rw[c0 + i] * id : 0.0;
    }
#pragma unroll
    for (int i = 0; i < B; ++i)
#pragma unroll
      for (int j = 0; j < B; ++j) v[i][j] = fma(-ri[i], rj[j], v[i][j]);
    if (k >= c0 && k < c0 + B) {
#pragma unroll
      for (int j = 0; j < B; ++j)
        if (c0 + j == k) {
#pragma unroll
          for (int i = 0; i < B; ++i)
            if (r0 + i >= k) v[i][j] = (r0 + i == k) ? d : ri[i];
        }
    }
  }
#pragma unroll
  for (int i = 0; i < B; ++i)
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const int gi = r0 + i, gj = c0 + j;
      if (gi < n && gj < n) a[gi * ld + gj] = (gj > gi) ? 0.0 : v[i][j];
    }
  __syncthreads();
  return ldl;
}

constexpr int kRC = 32;  // rows of B per chunk
constexpr int kLC = kMaxM + 1;  // LDS row stride of a chunk: consecutive rows start in different banks
static_assert(2 * kRC * kLC >= kMaxM * kMaxM, "the two chunk buffers hold an M x M matrix");

// The update and the projection for the forms that go on to invert L L' explicitly and keep its
// diagonal (the mean-field form, the EP cavity): rounding in W and L comes out multiplied by the
// condition of W (1e6 and more on a grid of 64 inducing points), so W is summed over the
// locations in their order and factored pivot by pivot, whatever the number of wavefronts.
// k_st_sites is faster (1.09 -> 0.45 ms at 4 runs of 500 steps, M = 64, R = 256) but rounds
// differently in the last place, which moved mean-field posteriors by 1e-9 to 5e-9.  Dense ones
// moved by 1e-14, infinite-horizon ones, which invert L L' too, by 2e-14 to 4e-13 (conditions of
// 3e3 to 7e5); against 80-bit arithmetic their errors are the same on both kernels, 7e-15 at a
// condition of 2e3, 3e-10 at 1e7, 1e-4 at 1e13.
// KIND: the likelihood as a compile-time constant (0: the projection, which has none);
// with only its branch compiled, the site step spills a fraction of what it does with
// every likelihood's code in the kernel.
template <int METHOD, int MODE, int KIND>
__global__ __launch_bounds__(kT, 3) void k_st_sites_ordered(StDims dm, LikParams lik, GHTable gh, StSiteIO io, double lr,
                                                 int ensure_psd, double power, int mask_pseudo) {
  extern __shared__ double smem[];
  if (KIND != 0) lik.kind = KIND;
  const int M = dm.M, R = dm.R;
  // LDS is kept near 53 KB (three workgroups per CU): the posterior covariance is read
  // from global memory by the GEMM, the projection W accumulates in its output slot Lw
  // (global, L2-resident) and comes into LDS (the chunk buffers) for the factorisation.
  double* pan = smem;                   // 2*kPK*kPS GEMM panels
  double* sC = pan + 2 * kPK * kPS;     // kRC rows of B (stride LC)
  double* sX = sC + kRC * kLC;          // kRC rows of B P, then nat2-scaled rows of B (stride LC)
  double* sW = sC;                      // M*M after the chunk loop (sC and sX together hold it)
  double* sm = sX + kRC * kLC;          // M posterior mean
  double* sv = sm + kMaxM;              // M: B' nat1 -> z
  double* sn = sv + kMaxM;              // kRC: new nat1 of the chunk
  double* row = sn + kRC;               // 2*kMaxM pivot rows
  double* red = row + 2 * kMaxM;        // 4
  const int t = blockIdx.x, k = blockIdx.y, tid = threadIdx.x;
  const int64_t kt = (int64_t)k * dm.T + t;
  const int LC = M + 1;
  constexpr bool UPDATE = MODE == BN_ST_UPDATE;
  constexpr bool SITES = MODE != BN_ST_PROJECT;
  const double* gP = io.pP + kt * M * M;
  double* gW = io.Lw + kt * M * M;
  // mini-batch (inference.py:65-90, group_natural_params basemodels.py:195-199): a step
  // outside it keeps its sites and adds no data term; its projection is still formed
  const bool in_batch = io.batch == nullptr || io.batch[kt] != 0.0f;
  if (SITES) {
    for (int e = tid; e < M; e += kT) sm[e] = io.pm[kt * M + e];
  }
  for (int e = tid; e < M; e += kT) sv[e] = 0.0;
  double acc0 = 0.0, acc1 = 0.0;
  for (int i0 = 0; i0 < R; i0 += kRC) {
    const int nr = min(kRC, R - i0);
    __syncthreads();
    for (int e = tid; e < kRC * M; e += kT) {
      const int i = e / M, j = e - i * M;
      sC[i * LC + j] = (e < nr * M) ? io.B[(kt * R + i0) * M + e] : 0.0;
    }
    if (SITES) {
      // X = C P ; row i: mean_f = c_i . m, var_f = c_i . x_i + diag C
      wg_gemm_small(kRC, M, M, 1.0, MatRef{sC, LC, 1}, MatRef{gP, M, 1}, 0.0, sX, LC, pan);
      if (tid < nr) {
        const int64_t s = kt * R + i0 + tid;
        double mf = 0.0, vf = io.cdiag[s];
        for (int j = 0; j < M; ++j) {
          const double c = sC[tid * LC + j];
          mf = fma(c, sm[j], mf);
          vf = fma(c, sX[tid * LC + j], vf);
        }
        const double yv = (double)io.y[s];
        if (!in_batch) {
        } else if (UPDATE) {
          const double n1 = io.nat1[s], n2 = io.nat2[s];
          // EP: (pm, pP) is the cavity of the inducing states, so (mf, vf) is the cavity at the data
          SiteResult sr = METHOD == M_EP ? ep_site_from_cavity(lik, gh, yv, mf, vf, power, mask_pseudo != 0,
                                                               ensure_psd != 0)
                                         : site_step<METHOD>(lik, gh, yv, mf, vf, n1, n2, 1.0, ensure_psd != 0);
          acc0 += fabs(sr.nat1 - n1);
          acc1 += fabs(sr.nat2 - n2);
          const double a1 = (1.0 - lr) * n1 + lr * sr.nat1, a2 = (1.0 - lr) * n2 + lr * sr.nat2;
          io.nat1[s] = a1;
          io.nat2[s] = a2;
          if (io.o_mean != nullptr) {
            io.o_mean[s] = (float)sr.mean;
            io.o_jac[s] = (float)sr.jac;
            io.o_hess[s] = (float)sr.hess;
          }
        }
      }
    }
    {
      __syncthreads();
      // X = diag(nat2) C (rows of the chunk), v += C' nat1, W += C' X
      for (int e = tid; e < kRC * M; e += kT) {
        const int i = e / M, j = e - i * M;
        sX[i * LC + j] = (i < nr) ? io.nat2[kt * R + i0 + i] * sC[i * LC + j] : 0.0;
      }
      if (tid < kRC) sn[tid] = (tid < nr) ? io.nat1[kt * R + i0 + tid] : 0.0;
      __syncthreads();
      if (tid < M) {
        double u = sv[tid];
        for (int i = 0; i < nr; ++i) u = fma(sC[i * LC + tid], sn[i], u);
        sv[tid] = u;
      }
      wg_gemm_small(M, M, kRC, 1.0, MatRef{sC, 1, LC}, MatRef{sX, LC, 1}, i0 == 0 ? 0.0 : 1.0, gW, M, pan);
    }
  }
  if (UPDATE) {
    const double d1 = wg_sum(acc0, red), d2 = wg_sum(acc1, red);
    if (tid == 0) { io.part0[kt] = d1; io.part1[kt] = d2; }
  }
  {
    __syncthreads();
    for (int e = tid; e < M * M; e += kT) sW[e] = gW[e] + ((e / M == e % M) ? kPseudoJitter : 0.0);
    const double ld = wg_chol_reg<kMaxM / 16>(sW, M, M, row);
    wg_lower_solve(sW, M, M, sv, 1, 0, 1);
    double* Lo = io.Lw + kt * M * M;
    for (int e = tid; e < M * M; e += kT) Lo[e] = sW[e];
    for (int e = tid; e < M; e += kT) io.zw[kt * M + e] = sv[e];
    if (tid == 0) io.ldl[kt] = ld;
  }
}

constexpr int kSLd = kMaxM + 2;  // row stride of the site kernel's LDS matrices
constexpr int kWT = 10;          // tiles (i, j <= i) of a 64 x 64 symmetric matrix

// Sums x[0..3] over the 16 lanes of a row of lanes; lane c of the row gets the sum of x[c / 4].
__device__ inline double row_sums4(const double (&x)[4], int l) {
  const bool h = l & 8, m = l & 4;
  double a = h ? x[2] : x[0], b = h ? x[3] : x[1];
  a += __shfl_xor(h ? x[0] : x[2], 8, 64);
  b += __shfl_xor(h ? x[1] : x[3], 8, 64);
  double s = m ? b : a;
  s += __shfl_xor(m ? a : b, 4, 64);
  s += __shfl_xor(s, 2, 64);
  s += __shfl_xor(s, 1, 64);
  return s;
}

// A L^-T for a row tile A, into X (row stride ld) and returned: the product with the explicit
// inverse I of the diagonal block, then one step of refinement with the block's factor L (row
// stride kSLd).  Without it L L' misses W by the condition of the diagonal blocks (16
// neighbouring inducing points) times the rounding unit.  That matters where W is singular but
// for its 1e-12: with 8 locations for 64 inducing points the remaining columns then lost their
// positive pivots and the factor became NaN.  With four locations an inducing point L L', the
// posteriors and the time (32 runs of 100 steps, 6.7 ms) are the same without it.
__device__ inline tile4 solve_tile(double* X, int ld, const double* I, const double* L, tile4 A, int l) {
  double a[4];
  tile_store(X, ld, 0, 0, A, l);
  wave_sync();
  tile4 v = tile_mul_t(X, ld, 0, I, kDiagLd, 0, 0, 0, tile_zero(), l);
  wave_sync();
  tile_store(X, ld, 0, 0, v, l);
  wave_sync();
  frag4(a, X, ld, 0, 0, -1.0, l);
#pragma unroll
  for (int c = 0; c < 4; ++c) A = mfma16(a[c], frag(L, kSLd, 0, 4 * c, l), A);
  wave_sync();
  tile_store(X, ld, 0, 0, A, l);
  wave_sync();
  v = tile_mul_t(X, ld, 0, I, kDiagLd, 0, 0, 0, v, l);
  wave_sync();
  tile_store(X, ld, 0, 0, v, l);
  wave_sync();
  return v;
}

// KIND: the likelihood as a compile-time constant (0: the projection, which has none).
//
// A wavefront works through 16 rows of B at a time on its own: X = C P with P's lower tiles only
// (diag(C P C') = sum_j C_ij (C_j P_jj + 2 sum_k>j C_k P_kj)_ij), the site step of the 16
// locations, and its share of the lower tiles of W = B' diag(nat2) B in registers; the four
// wavefronts meet for the sum of W and its blocked Cholesky factorisation (chol16_inverse).
// 71 KB of LDS, two workgroups a CU, so that one's factorisation runs under the other's
// products.  Bound by the FP64 matrix instructions (20 k cycles a SIMD a step at M = 64, R = 256)
// and the four pivot chains.
template <int METHOD, int MODE, int KIND>
__global__ __launch_bounds__(kT, 2) void k_st_sites(StDims dm, LikParams lik, GHTable gh, StSiteIO io, double lr,
                                                 int ensure_psd, double power, int mask_pseudo) {
  extern __shared__ double smem[];
  if (KIND != 0) lik.kind = KIND;
  const int M = dm.M, R = dm.R, MB = (M + 15) / 16;
  double* sP = smem;                      // kMaxM x kSLd: posterior covariance; partial sums of W; Lm
  double* sB = sP + kMaxM * kSLd;         // 4 x 16 x kSLd: the wavefronts' rows of B; partial sums of W; L (ENERGY)
  double* sI = sB;                        // 4 x 16 x kDiagLd: diagonal blocks, then their inverse factors
  double* sG = sI + 4 * 16 * kDiagLd;     // 16 x kDiagLd: row tile of v' (both once W is summed)
  double* sm = sB + kMaxM * kSLd;         // kMaxM: posterior mean
  double* sv = sm + kMaxM;                // 4 x kMaxM: the wavefronts' parts of v = B' nat1; z
  double* sn = sv + 4 * kMaxM;            // 4 x 2 x 16: new nat1, nat2 of the wavefronts' rows
  double* red = sn + 4 * 32;              // 4
  const int t = blockIdx.x, k = blockIdx.y, tid = threadIdx.x;
  int l = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t kt = (int64_t)k * dm.T + t;
  constexpr bool UPDATE = MODE == BN_ST_UPDATE;
  constexpr bool PROJECT = MODE != BN_ST_ENERGY;
  constexpr bool SITES = MODE != BN_ST_PROJECT;
  // mini-batch (inference.py:65-90, group_natural_params basemodels.py:195-199): a step
  // outside it keeps its sites and adds no data term; its projection is still formed
  const bool in_batch = io.batch == nullptr || io.batch[kt] != 0.0f;
  double* cB = sB + w * 16 * kSLd;
  double* cn = sn + w * 32;
  const int RT = (R + 15) / 16;
  double pre[16];  // the next 16 rows of B, one column a lane
  auto fetch = [&](int rt) {
    const double* src = io.B + (kt * R + 16 * rt) * M + l;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      pre[i] = *(l < M && 16 * rt + i < R ? src + i * M : io.B);  // masked when it is placed
    }
  };
  if (w < RT) fetch(w);
  if (SITES) {
    const double* gP = io.pP + kt * M * M;
#pragma unroll 4
    for (int i = w; i < 16 * MB; i += 4) sP[i * kSLd + l] = (i < M && l < M) ? gP[i * M + l] : 0.0;
    if (tid < kMaxM) sm[tid] = tid < M ? io.pm[kt * M + tid] : 0.0;
  }
  __syncthreads();
  tile4 W[kWT];
  double va[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int i = 0; i < kWT; ++i) W[i] = tile_zero();
  double acc0 = 0.0, acc1 = 0.0;
#pragma unroll 1
  for (int rt = w; rt < RT; rt += 4) {
    l = fresh_v(l);
    wave_sync();
#pragma unroll
    for (int i = 0; i < 16; ++i) cB[i * kSLd + l] = l < M && 16 * rt + i < R ? pre[i] : 0.0;
    // the lane's location in the site step: row l/16 + 4 ((l%16) / 4), the first of four lanes writes
    const int row = (l >> 4) + (l & 12), at = 16 * rt + row;
    const bool mine = (l & 3) == 0 && at < R;
    const int64_t s = kt * R + (at < R ? at : 0);
    double n1 = 0.0, n2 = 0.0, cd = 0.0, yv = 0.0;
    if (MODE != BN_ST_ENERGY) {
      n1 = io.nat1[s];
      n2 = io.nat2[s];
    }
    if (SITES) {
      cd = io.cdiag[s];
      yv = (double)io.y[s];
    }
    if (rt + 4 < RT) fetch(rt + 4);
    wave_sync();
    if (SITES) {
      tile4 X[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) X[j] = tile_zero();
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        if (kk < MB) {
          double a[4];
          frag4(a, cB, kSLd, 0, 16 * kk, 1.0, l);
#pragma unroll
          for (int c = 0; c < 4; ++c) X[kk] = mfma16(a[c], frag(sP, kSLd, 16 * kk, 16 * kk + 4 * c, l), X[kk]);
#pragma unroll
          for (int j = 0; j < kk; ++j)
#pragma unroll
            for (int c = 0; c < 4; ++c) X[j] = mfma16(2.0 * a[c], frag(sP, kSLd, 16 * j, 16 * kk + 4 * c, l), X[j]);
        }
      double mq[4] = {0.0, 0.0, 0.0, 0.0}, vq[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j < MB) {
          const double mj = sm[16 * j + (l & 15)];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const double c = cB[((l >> 4) + 4 * q) * kSLd + 16 * j + (l & 15)];
            mq[q] = fma(c, mj, mq[q]);
            vq[q] = fma(c, X[j][q], vq[q]);
          }
        }
      const double mf = row_sums4(mq, l), vf = cd + row_sums4(vq, l);
      if (!in_batch || !mine) {
      } else if (UPDATE) {
        static_assert(!UPDATE || METHOD != M_EP, "the EP update goes through k_st_sites_ordered");
        const SiteResult sr = site_step<METHOD>(lik, gh, yv, mf, vf, n1, n2, 1.0, ensure_psd != 0);
        acc0 += fabs(sr.nat1 - n1);
        acc1 += fabs(sr.nat2 - n2);
        n1 = (1.0 - lr) * n1 + lr * sr.nat1;
        n2 = (1.0 - lr) * n2 + lr * sr.nat2;
        io.nat1[s] = n1;
        io.nat2[s] = n2;
        if (io.o_mean != nullptr) {
          io.o_mean[s] = (float)sr.mean;
          io.o_jac[s] = (float)sr.jac;
          io.o_hess[s] = (float)sr.hess;
        }
      } else if (METHOD == M_EP) {
        acc0 += ep_lel_from_cavity(lik, gh, yv, mf, vf, power);
      } else {
        double t1, t2;
        energy_terms<METHOD>(lik, gh, yv, mf, vf, 1.0, 1.0, 1.0, t1, t2);
        acc0 += t1;
      }
    }
    if (PROJECT) {
      if ((l & 3) == 0) {
        cn[row] = at < R ? n1 : 0.0;
        cn[16 + row] = at < R ? n2 : 0.0;
      }
      wave_sync();
#pragma unroll
      for (int c = 0; c < 16; c += 4) {
        const double e1 = cn[c + (l >> 4)], e2 = cn[16 + c + (l >> 4)];
        double f[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          f[j] = j < MB ? frag_t(cB, kSLd, c, 16 * j, l) : 0.0;
          va[j] = fma(f[j], e1, va[j]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (i < MB) {
#pragma unroll
            for (int j = 0; j <= i; ++j) W[i * (i + 1) / 2 + j] = mfma16(f[i], e2 * f[j], W[i * (i + 1) / 2 + j]);
          }
      }
    }
  }
  if (UPDATE) {
    const double d1 = wg_sum(acc0, red), d2 = wg_sum(acc1, red);
    if (tid == 0) { io.part0[kt] = d1; io.part1[kt] = d2; }
  }
  if (PROJECT) {
    // sum of the wavefronts' parts: 0 + 2 and 1 + 3, then the two
    constexpr int kPart = kWT * 256;
    static_assert(2 * kPart <= 2 * kMaxM * kSLd, "two partial sums of W fit the covariance's and the rows' space");
    __syncthreads();
    l = fresh_v(l);
    double* part = sP + (w & 1) * kPart;
    if (w >= 2) {
#pragma unroll
      for (int i = 0; i < kWT; ++i) tile_put(part + i * 256, W[i], l);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      va[j] += __shfl_xor(va[j], 16, 64);
      va[j] += __shfl_xor(va[j], 32, 64);
      if (l < 16) sv[w * kMaxM + 16 * j + l] = va[j];
    }
    __syncthreads();
    if (w < 2) {
#pragma unroll
      for (int i = 0; i < kWT; ++i) {
        W[i] += tile_get(part + i * 256, l);
        tile_put(part + i * 256, W[i], l);
      }
    }
    __syncthreads();
    // row tile w of W + 1e-12 I (identity padding); wavefront 0 also takes v' as a row tile
    tile4 V[4], Z[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      V[j] = tile_zero();
      Z[j] = tile_zero();
      if (j <= w && w < MB) {
        const int o = (w * (w + 1) / 2 + j) * 256;
        V[j] = tile_get(sP + o, l) + tile_get(sP + kPart + o, l);
      }
      const int e = 16 * j + (l & 15);
      if (w == 0) Z[j][0] = l < 16 ? (sv[e] + sv[2 * kMaxM + e]) + (sv[kMaxM + e] + sv[3 * kMaxM + e]) : 0.0;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (j == w && (l >> 4) + 4 * q == (l & 15)) V[j][q] += e < M ? kPseudoJitter : 1.0;
    }
    __syncthreads();
    double* Lm = sP;
    for (int e = tid; e < 16 * kDiagLd; e += kT) sG[e] = 0.0;
    if (w == 0) {
      tile_store(sI, kDiagLd, 0, 0, V[0], l);
      wave_sync();
      chol16_inverse<true>(sI, kDiagLd, l, Lm, kSLd);
    }
#pragma unroll 1
    for (int b = 0; b < MB; ++b) {
      const double* Ib = sI + b * 16 * kDiagLd;
      __syncthreads();  // inverse factor of diagonal block b
      l = fresh_v(l);
      if (w > b && w < MB) {
        solve_tile(Lm + 16 * w * kSLd + 16 * b, kSLd, Ib, Lm + 16 * b * kSLd + 16 * b, V[0], l);
        if (w == b + 1) {  // the next diagonal block first
          double a[4];
          frag4(a, Lm, kSLd, 16 * w, 16 * b, 1.0, l);
#pragma unroll
          for (int c = 0; c < 4; ++c) V[1] = mfma16(-a[c], a[c], V[1]);
          tile_store(sI + (b + 1) * 16 * kDiagLd, kDiagLd, 0, 0, V[1], l);
        }
      } else if (w == 0) {
        const tile4 v = solve_tile(sG, kDiagLd, Ib, Lm + 16 * b * kSLd + 16 * b, Z[0], l);
        if (l < 16) sm[16 * b + l] = v[0];  // z
      }
      __syncthreads();  // column block b of Lm
      l = fresh_v(l);
      if (b + 1 < MB) {
        if (w == b + 1) {
          chol16_inverse<true>(sI + w * 16 * kDiagLd, kDiagLd, l, Lm + 16 * w * kSLd + 16 * w, kSLd);
        } else if ((w > b + 1 && w < MB) || w == 0) {
          double a[4];
          frag4(a, w == 0 ? sG : Lm + 16 * w * kSLd + 16 * b, w == 0 ? kDiagLd : kSLd, 0, 0, -1.0, l);
#pragma unroll
          for (int j = 1; j < 4; ++j)
            if (b + j < MB) {
#pragma unroll
              for (int c = 0; c < 4; ++c) {
                const double f = frag(Lm, kSLd, 16 * (b + j), 16 * b + 4 * c, l);
                if (w == 0) Z[j] = mfma16(a[c], f, Z[j]);
                else V[j] = mfma16(a[c], f, V[j]);
              }
            }
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) { V[j] = V[j + 1]; Z[j] = Z[j + 1]; }
      }
    }
    __syncthreads();
    double* Lo = io.Lw + kt * M * M;
    for (int i = w; i < M; i += 4)
      if (l < M) Lo[i * M + l] = (l >> 4) > (i >> 4) ? 0.0 : Lm[i * kSLd + l];
    if (tid < M) io.zw[kt * M + tid] = sm[tid];
    if (w == 3) {
      double ld = l < M ? -log(sI[(l >> 4) * 16 * kDiagLd + (l & 15) * (kDiagLd + 1)]) : 0.0;
      for (int o = 32; o > 0; o >>= 1) ld += __shfl_xor(ld, o, 64);
      if (l == 0) io.ldl[kt] = ld;
    }
  } else if (METHOD == M_EP) {
    // the pseudo term (lel_pseudo) comes from k_st_ep_cavity
    const double e1 = wg_sum(acc0, red);
    if (tid == 0) io.part0[kt] = e1;
  } else {
    // whitened expected density of the pseudo observation:
    // |z - L' m|^2 and tr(L' P L) = sum_ac L(a,c) (P L)(a,c)
    const double* L = io.Lw + kt * M * M;
    const double e1 = wg_sum(acc0, red);  // every wavefront has read its rows of B
#pragma unroll 4
    for (int i = w; i < 16 * MB; i += 4) sB[i * kSLd + l] = (i < M && l < M) ? L[i * M + l] : 0.0;
    __syncthreads();
    l = fresh_v(l);
    double q2 = 0.0, tr = 0.0;
    if (tid < M) {
      double u = io.zw[kt * M + tid];
#pragma unroll 4
      for (int a = tid; a < M; ++a) u = fma(-sB[a * kSLd + tid], sm[a], u);  // (z - L' m)_tid
      q2 = u * u;
    }
    if (w < MB) {
      tile4 X[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) X[j] = tile_zero();
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        if (kk < MB) {
#pragma unroll
          for (int c = 0; c < 16; c += 4) {
            const double a = frag(sP, kSLd, 16 * w, 16 * kk + c, l);
#pragma unroll
            for (int j = 0; j <= kk; ++j) X[j] = mfma16(a, frag_t(sB, kSLd, 16 * kk + c, 16 * j, l), X[j]);
          }
        }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j < MB) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            tr = fma(sB[(16 * w + (l >> 4) + 4 * q) * kSLd + 16 * j + (l & 15)], X[j][q], tr);
        }
    }
    const double Q2 = wg_sum(q2, red), TR = wg_sum(tr, red);
    if (tid == 0) {
      io.part0[kt] = e1;
      io.part1[kt] = -0.5 * (Q2 + M * kLog2Pi - 2.0 * io.ldl[kt]) - 0.5 * TR;
    }
  }
}

// ---------------------------------------------------------------------------
// k_st_ep_cavity: per (step, run), the power-EP cavity of the inducing states
// (compute_cavity, utils.py:534-541, on the projected sites of basemodels.py:667-674):
//   Q = P + 1e-8 I,  W = B' diag(nat2) B = L L' - 1e-12 I  (L, z from the projection),
//   cav_cov = (Q^-1 - a W)^-1,  cav_mean = cav_cov (Q^-1 m - a B' nat1),  B' nat1 = L z.
// ENERGY also forms the pseudo term of the EP energy (basemodels.py:247-262),
//   lel_pseudo = log N(py | cav_mean, pv / a + cav_cov) + pep_constant(pv, a),
// with pv = (W + 1e-12 I)^-1 and py = pv B' nat1, in whitened form: w = z - L' cav_mean,
// G = I / a + L' cav_cov L, log N = -1/2 (w' G^-1 w + M log 2pi - 2 log|L| + log|G|),
// pep_constant = M/2 ((1 - a) log 2pi - log a) - (1 - a) log|L|; so pv, whose
// eigenvalues reach 1e12, is never formed.  mask_pseudo with a missing output at a
// one-location step: 0 (mvn_logpdf and pep_constant of a fully masked observation).
// ---------------------------------------------------------------------------
struct StCavityIO {
  const float* y;      // [K,T,R]
  const double* pm;    // [K,T,M]
  const double* pP;    // [K,T,M,M]
  const double* Lw;    // [K,T,M,M]
  const double* zw;    // [K,T,M]
  const double* ldl;   // [K,T]
  double* cm;          // [K,T,M]
  double* cP;          // [K,T,M,M]
  double* lel_pseudo;  // [K,T] (ENERGY)
};

template <bool ENERGY>
__global__ __launch_bounds__(kT) void k_st_ep_cavity(StDims dm, StCavityIO io, double power, int mask_pseudo) {
  extern __shared__ double smem[];
  const int M = dm.M;
  double* pan = smem;                    // 2*kPK*kPS
  double* sQ = pan + 2 * kPK * kPS;      // M*M
  double* sA = sQ + kMaxM * kMaxM;       // M*M
  double* sm = sA + kMaxM * kMaxM;       // M: posterior mean, then cav_mean
  double* sr = sm + kMaxM;               // M: right-hand side, then w
  double* row = sr + kMaxM;              // 2*kMaxM pivot rows
  double* red = row + 2 * kMaxM;         // 4
  const int t = blockIdx.x, k = blockIdx.y, tid = threadIdx.x;
  const int64_t kt = (int64_t)k * dm.T + t;
  const double* P = io.pP + kt * M * M;
  const double* L = io.Lw + kt * M * M;
  const double* z = io.zw + kt * M;
  for (int e = tid; e < M * M; e += kT) sQ[e] = P[e] + ((e / M == e % M) ? 1e-8 : 0.0);
  for (int e = tid; e < M; e += kT) sm[e] = io.pm[kt * M + e];
  wg_sweep_inv<kMaxM / 16, false>(sQ, M, M, row);                          // sQ = -Q^-1
  wg_gemm_small(M, M, M, 1.0, MatRef{L, M, 1}, MatRef{L, 1, M}, 0.0, sA, M, pan);  // L L'
  for (int e = tid; e < M * M; e += kT)
    sA[e] = -sQ[e] - power * sA[e] + ((e / M == e % M) ? power * kPseudoJitter : 0.0);
  if (tid < M) {
    double u = 0.0;
    for (int j = 0; j < M; ++j) u = fma(-sQ[tid * M + j], sm[j], u);
    for (int j = 0; j <= tid; ++j) u = fma(-power * L[tid * M + j], z[j], u);
    sr[tid] = u;
  }
  wg_sweep_inv<kMaxM / 16, false>(sA, M, M, row);                          // sA = -cav_cov
  double cmv = 0.0;
  if (tid < M) {
    for (int j = 0; j < M; ++j) cmv = fma(-sA[tid * M + j], sr[j], cmv);
    io.cm[kt * M + tid] = cmv;
  }
  double* gC = io.cP + kt * M * M;
  for (int e = tid; e < M * M; e += kT) gC[e] = -sA[e];
  if (!ENERGY) return;
  __syncthreads();
  if (tid < M) sm[tid] = cmv;
  __syncthreads();
  if (tid < M) {
    double u = z[tid];
    for (int a = tid; a < M; ++a) u = fma(-L[a * M + tid], sm[a], u);
    sr[tid] = u;                                                             // w = z - L' cav_mean
  }
  wg_gemm_small(M, M, M, -1.0, MatRef{sA, M, 1}, MatRef{L, M, 1}, 0.0, sQ, M, pan);  // cav_cov L
  wg_gemm_small(M, M, M, 1.0, MatRef{L, 1, M}, MatRef{sQ, M, 1}, 0.0, sA, M, pan);   // L' cav_cov L
  for (int e = tid; e < M * M; e += kT)
    if (e / M == e % M) sA[e] += 1.0 / power;
  const double ldg = wg_sweep_inv<kMaxM / 16, true>(sA, M, M, row);       // sA = -G^-1
  double q = 0.0;
  if (tid < M) {
    double u = 0.0;
    for (int j = 0; j < M; ++j) u = fma(-sA[tid * M + j], sr[j], u);
    q = sr[tid] * u;
  }
  const double Q2 = wg_sum(q, red);
  if (tid == 0) {
    const double ldl = io.ldl[kt];
    const double lp = -0.5 * (Q2 + M * kLog2Pi - 2.0 * ldl + ldg);
    const double pep = 0.5 * M * ((1.0 - power) * kLog2Pi - log(power)) - (1.0 - power) * ldl;
    const bool masked = mask_pseudo != 0 && dm.R == 1 && io.y[kt] != io.y[kt];
    io.lel_pseudo[kt] = masked ? 0.0 : lp + pep;
  }
}

// ---------------------------------------------------------------------------
// k_st_marginals: q(f) at every data location, mean_f = B m, var_f = diag(B P B') + diag C
// (conditional_posterior_to_data, basemodels.py:743-764, diagonal only).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kT) void k_st_marginals(StDims dm, const double* __restrict__ B,
                                                     const double* __restrict__ cdiag, const double* __restrict__ pm,
                                                     const double* __restrict__ pP, double* __restrict__ mean_f,
                                                     double* __restrict__ var_f) {
  __shared__ double sP[kMaxM * kMaxM];
  __shared__ double sm[kMaxM];
  const int M = dm.M, R = dm.R;
  const int t = blockIdx.x, k = blockIdx.y, tid = threadIdx.x;
  const int64_t kt = (int64_t)k * dm.T + t;
  for (int e = tid; e < M * M; e += kT) sP[e] = pP[kt * M * M + e];
  for (int e = tid; e < M; e += kT) sm[e] = pm[kt * M + e];
  __syncthreads();
  for (int i = tid; i < R; i += kT) {
    const int64_t s = kt * R + i;
    const double* b = B + s * M;
    double mf = 0.0, vf = cdiag[s];
    for (int j = 0; j < M; ++j) {
      const double bj = b[j];
      mf = fma(bj, sm[j], mf);
      double u = 0.0;
      for (int q = 0; q < M; ++q) u = fma(sP[j * M + q], b[q], u);
      vf = fma(bj, u, vf);
    }
    mean_f[s] = mf;
    var_f[s] = vf;
  }
}

// ---------------------------------------------------------------------------
// k_st_transitions: A(dt_t), Q(dt_t) of every (step, run), 2 KT^2 values each, so that the
// recursions read them as uniform values instead of evaluating them on one lane per step.
// ---------------------------------------------------------------------------
template <int KT>
__global__ __launch_bounds__(kT) void k_st_transitions(StDims dm, StHyp hy, const double* __restrict__ dt,
                                                       double* __restrict__ aq) {
  const int64_t e = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (e >= (int64_t)dm.K * dm.T) return;
  const int64_t k = e / dm.T;
  double A[KT * KT], Q[KT * KT];
  temporal_AQ<KT>(hy.ls_t[k * hy.stride], hy.var_t[k * hy.stride], dt[e], A, Q);
  double* o = aq + e * 2 * KT * KT;
  for (int i = 0; i < KT * KT; ++i) { o[i] = A[i]; o[KT * KT + i] = Q[i]; }
}

// ---------------------------------------------------------------------------
// k_st_filter: one workgroup per run, sequential over T (ops.py:154-180 in whitened form).
// Per step, with U = P-[:, :M] L and the Cholesky factor Lm Lm' = Mm = I + L' U[:M]:
//   W = U Lm^-T,  e = Lm^-1 (z - L' H m-),  m = m- + W e,  P = P- - W W',
//   log N = -1/2 (e' e + M log 2pi + log det Mm - 2 ldl).
//
// Bound by the latency of one workgroup's chain of steps.  At M = 64, D = 128 a step has 23 k
// cycles of FP64 matrix instructions a SIMD (64 cycles each) and four pivot chains of 3.5 k
// cycles; it takes 61 k cycles = 25 us, against 126 us for products from L2 through LDS panels
// with a 64-pivot sweep inverse (one run of 1000 steps: 125.6 -> 25 ms).
// The covariance stays in registers for the whole walk: a wavefront holds the 16 x 16 tiles
// (i, j), i <= j, of all KT x KT blocks, so the predict step, which mixes blocks elementwise,
// touches no memory, and the tiles below the diagonal are transposes of held ones.  Predict
// and W W' round alike for an entry and its mirror image, so the diagonal tiles stay
// symmetric to the last bit.  [Mm; U; q'] is eliminated together, 16 columns at a
// time: one wavefront factors the diagonal block (chol16_inverse), every wavefront multiplies
// its row tiles by the block's inverse, then updates its remaining columns and its part of P
// while the next diagonal block is factored.  M is padded to 16 MB with zero rows of L, which
// leave Mm's padding the identity.
// ---------------------------------------------------------------------------
struct StFilterIO {
  const double* aq;   // [K,T,2 KT^2] transitions
  const double* Lw;   // [K,T,M,M]
  const double* zw;   // [K,T,M]
  double* fmean;      // [K,T,D] filtered means
  double* fcov;       // [K,T,D(D+1)/2] filtered covariances, packed upper triangle by rows
  double* ell;        // [K,T] per-step log-likelihood terms: e' e, until k_st_ell completes them
  double* det;        // [K,T,2] mantissa and exponent of 1 / sqrt(det Mm)
};

// ell = -1/2 (e' e + M log 2pi + log det Mm - 2 ldl), one step a thread: the logarithms stay
// out of the recursion.
__global__ __launch_bounds__(kT) void k_st_ell(StDims dm, const double* __restrict__ det,
                                               const double* __restrict__ ldl, double* __restrict__ ell) {
  const int64_t e = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (e >= (int64_t)dm.K * dm.T) return;
  const double ld = -2.0 * (log(det[2 * e]) + det[2 * e + 1] * 0.69314718055994530942);
  ell[e] = -0.5 * (ell[e] + dm.M * kLog2Pi + ld - 2.0 * ldl[e]);
}

// packed upper-triangle index of (i, j), i <= j, in an n x n matrix
__device__ inline int64_t pidx(int i, int j, int n) { return (int64_t)i * n - (int64_t)i * (i - 1) / 2 + (j - i); }

// LDS of k_st_filter in doubles
constexpr int filter_smem(int KT, int MB) {
  const int MP = 16 * MB, LD = MP + 2;
  return (KT + 2) * MP * LD + (MB + 1) * 16 * kDiagLd + 2 * MP + KT * MP + 2 * KT * KT;
}

// The covariance P of a state of KT components of MP = 16 MB entries in registers (the tiles
// (i, j), i <= j, of its KT x KT blocks), and its update P -= W W' with W = U Lm^-T from the blocked
// elimination of [Mm; U; q'].
template <int KT, int MB>
struct FilterCore {
  static constexpr int MP = 16 * MB, LD = MP + 2, NW = 2 * MB, NT = 64 * NW;
  static constexpr int NR = KT * MB;                  // row tiles of U
  static constexpr int NPOS = MB * (MB + 1) / 2;      // tile positions of P
  static constexpr int NP = (NPOS + NW - 1) / NW;     // positions per wavefront, at most
  static constexpr bool kAllR = NR == NW;
  typedef tile4 Cov[NP][KT][KT];

  // position n of wavefront w: w, then (four tiles a side only, 10 positions) 8 on wavefront 0 and
  // 9 on wavefront 6, whose SIMDs are not the ones that factor the second and the last block
  static __device__ inline bool position(int w, int n, int& i, int& j) {
    int p = n == 0 ? w : (w == 0 ? 8 : w == 6 ? 9 : NPOS);
    const bool on = p < NPOS;
    i = 0;
#pragma unroll
    for (int r = 0; r < MB - 1; ++r)
      if (i == r && p >= MB - r) { p -= MB - r; i = r + 1; }
    j = i + p;
    return on;
  }

  // P := (A (x) I) P (A (x) I)' + Q (x) I; the mixed products are added first, so that an entry and
  // its mirror image round alike
  static __device__ inline void predict(Cov& P, const double (&A)[KT][KT], const double (&Q)[KT][KT], int M, int w,
                                        int l) {
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      int i, j;
      if (!position(w, n, i, j)) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int gi = 16 * i + (l >> 4) + 4 * q, gj = 16 * j + (l & 15);
        const double on = gi == gj && gi < M ? 1.0 : 0.0;
        if (KT == 1) {
          P[n][0][0][q] = fma(A[0][0] * A[0][0], P[n][0][0][q], on * Q[0][0]);
        } else {
          constexpr int o = KT - 1;
          const double a = P[n][0][0][q], b = P[n][0][o][q], c = P[n][o][0][q], d = P[n][o][o][q];
          const double s = b + c;
          P[n][0][0][q] = fma(A[0][0] * A[0][0], a, fma(A[0][0] * A[0][o], s, fma(A[0][o] * A[0][o], d, on * Q[0][0])));
          P[n][o][o][q] = fma(A[o][0] * A[o][0], a, fma(A[o][0] * A[o][o], s, fma(A[o][o] * A[o][o], d, on * Q[o][o])));
          const double u = fma(A[0][0] * A[o][0], a, fma(A[0][o] * A[o][o], d, on * Q[0][o]));
          const double x = A[0][0] * A[o][o], y = A[0][o] * A[o][0];
          P[n][0][o][q] = fma(y, c, fma(x, b, u));
          P[n][o][0][q] = fma(y, b, fma(x, c, u));
        }
      }
    }
  }

  // X := P[:, :M]
  static __device__ inline void publish(const Cov& P, double* X, int w, int l) {
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      int i, j;
      if (!position(w, n, i, j)) continue;
#pragma unroll
      for (int a = 0; a < KT; ++a) {
        tile_store(X, LD, (a * MB + i) * 16, 16 * j, P[n][a][0], l);
        if (i != j) tile_store_t(X, LD, (a * MB + j) * 16, 16 * i, P[n][0][a], l);
      }
    }
  }

  static __device__ inline void update(Cov& P, const double* X, int b, int w, int l) {  // P -= W_b W_b'
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      int i, j;
      if (!position(w, n, i, j)) continue;
#pragma unroll
      for (int c = 0; c < 16; c += 4) {
        double ra[KT], rb[KT];
#pragma unroll
        for (int a = 0; a < KT; ++a) {
          ra[a] = -frag(X, LD, (a * MB + i) * 16, 16 * b + c, l);
          rb[a] = frag(X, LD, (a * MB + j) * 16, 16 * b + c, l);
        }
#pragma unroll
        for (int a = 0; a < KT; ++a)
#pragma unroll
          for (int d = 0; d < KT; ++d) P[n][a][d] = mfma16(ra[a], rb[d], P[n][a][d]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // The elimination.  U: row tile w of U (also in X); V: row tile w of Mm (w < MB, column tiles
  // <= w) or, with QROW, q' (the last wavefront); the first diagonal block's inverse factor is in sI
  // (wavefront 0).  X: U in, W out; se: e, quad: e' e in the lanes of the last wavefront.
  // One copy of the block's code: U and V are shifted by one tile after each block, so that tile 0
  // is always the current one.
  template <bool QROW>
  static __device__ inline void eliminate(Cov& P, tile4 (&U)[MB], tile4 (&V)[MB], double& quad, double* X, double* Lm,
                                          double* sI, double* sG, double* se, const int w0, const int tid0) {
    int w = w0, l = tid0 & 63;
    auto phase = [&]() { w = fresh_s(w0); l = fresh_v(tid0) & 63; };
#pragma unroll 1
    for (int b = 0; b < MB; ++b) {
      const double* Ib = sI + b * 16 * kDiagLd;
      __syncthreads();  // inverse factor of diagonal block b
      phase();
      // row tiles times the inverse factor's transpose: column block b of W, Lm and e
      if (w > b && w < MB) {
        tile_store(Lm, LD, 16 * w, 16 * b, V[0], l);
        wave_sync();
        const tile4 v = tile_mul_t(Lm, LD, 16 * w, Ib, kDiagLd, 0, 16 * b, 0, tile_zero(), l);
        wave_sync();
        tile_store(Lm, LD, 16 * w, 16 * b, v, l);
      } else if (QROW && w == NW - 1) {
        tile_store(sG, kDiagLd, 0, 0, V[0], l);
        wave_sync();
        const tile4 v = tile_mul_t(sG, kDiagLd, 0, Ib, kDiagLd, 0, 0, 0, tile_zero(), l);
        wave_sync();
        tile_store(sG, kDiagLd, 0, 0, v, l);
        if (l < 16) {
          se[16 * b + l] = v[0];
          quad = fma(v[0], v[0], quad);
        }
      }
      if (kAllR || w < NR) {
        if (b > 0) {
          tile_store(X, LD, 16 * w, 16 * b, U[0], l);
          wave_sync();
        }
        const tile4 v = tile_mul_t(X, LD, 16 * w, Ib, kDiagLd, 0, 16 * b, 0, tile_zero(), l);
        wave_sync();
        tile_store(X, LD, 16 * w, 16 * b, v, l);
      }
      if (MB > 1 && w == b + 1 && w < MB) {
        // the next diagonal block first: its factorisation is the critical path
#pragma unroll
        for (int c = 0; c < 16; c += 4) {
          const double a = frag(Lm, LD, 16 * w, 16 * b + c, l);
          V[MB > 1 ? 1 : 0] = mfma16(-a, a, V[MB > 1 ? 1 : 0]);
        }
        tile_store(sI + (b + 1) * 16 * kDiagLd, kDiagLd, 0, 0, V[MB > 1 ? 1 : 0], l);
      }
      __syncthreads();  // column block b of W and Lm
      phase();
      // remaining columns of the row tiles
      if (b + 1 < MB) {
        if (w == b + 1) chol16_inverse(sI + (b + 1) * 16 * kDiagLd, kDiagLd, l);
        double a[4];
        const bool qrow = QROW && w == NW - 1;
        if ((w > b + 1 && w < MB) || qrow) {
          const double* S = qrow ? sG : Lm + 16 * w * LD + 16 * b;
          const int ld = qrow ? kDiagLd : LD;
#pragma unroll
          for (int c = 0; c < 4; ++c) a[c] = -frag(S, ld, 0, 4 * c, l);
#pragma unroll
          for (int j = 1; j < MB; ++j)
            if (b + j < MB) {
#pragma unroll
              for (int c = 0; c < 4; ++c) V[j] = mfma16(a[c], frag(Lm, LD, 16 * (b + j), 16 * b + 4 * c, l), V[j]);
            }
        }
        if (kAllR || w < NR) {
#pragma unroll
          for (int c = 0; c < 4; ++c) a[c] = -frag(X, LD, 16 * w, 16 * b + 4 * c, l);
#pragma unroll
          for (int j = 1; j < MB; ++j)
            if (b + j < MB) {
#pragma unroll
              for (int c = 0; c < 4; ++c) U[j] = mfma16(a[c], frag(Lm, LD, 16 * (b + j), 16 * b + 4 * c, l), U[j]);
            }
        }
#pragma unroll
        for (int j = 0; j + 1 < MB; ++j) { U[j] = U[j + 1]; V[j] = V[j + 1]; }
      }
      // (a wavefront on the SIMD that factors the next block leaves its part to the last one)
      const int late = (w & 3) > 0 && (w & 3) < MB ? (w & 3) - 1 : -1;
      const int n = b == late ? 0 : b == MB - 1 && late >= 0 ? 2 : 1;
#pragma unroll 1
      for (int u = 0; u < n; ++u) update(P, X, u == 0 ? b : late, w, l);
    }
  }
};

// Row tile I of the lower triangle of Mm = I + L' U[:M] (column tiles <= I; L' is upper
// triangular, so inner tiles >= I).
template <int MB, int I>
__device__ inline void filter_mm_row(const double* LT, const double* X, int ld, tile4 (&V)[MB], int l) {
#pragma unroll
  for (int j = 0; j <= I; ++j) V[j] = tile_zero();
#pragma unroll
  for (int q = 0; q < 4; ++q) V[I][q] = (l >> 4) + 4 * q == (l & 15) ? 1.0 : 0.0;
#pragma unroll
  for (int kk = I; kk < MB; ++kk) {
#pragma unroll
    for (int c = 0; c < 16; c += 4) {
      const double a = frag(LT, ld, 16 * I, 16 * kk + c, l);
#pragma unroll
      for (int j = 0; j <= I; ++j) V[j] = mfma16(a, frag_t(X, ld, 16 * kk + c, 16 * j, l), V[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <int KT, int MB>
__global__ __launch_bounds__(128 * MB, 2) void k_st_filter(StDims dm, StHyp hy, StFilterIO io) {
  using C = FilterCore<KT, MB>;
  constexpr int MP = C::MP, LD = C::LD, NW = C::NW, NT = C::NT, NR = C::NR, NP = C::NP;
  constexpr bool kAllR = C::kAllR;
  constexpr int NL = (MP * MP + NT - 1) / NT;       // elements of L per thread
  constexpr int NAQ = 2 * KT * KT;
  extern __shared__ double smem[];
  double* X = smem;                    // KT*MP x LD: P-[:, :M], then U, then W
  double* LT = X + KT * MP * LD;       // MP x LD: L'
  double* Lm = LT + MP * LD;           // MP x LD: Lm below the diagonal blocks
  double* sI = Lm + MP * LD;           // MB of 16 x kDiagLd: diagonal blocks, then their inverse factors
  double* sG = sI + MB * 16 * kDiagLd; // 16 x kDiagLd: row tile of q'
  double* sq = sG + 16 * kDiagLd;      // MP: z, then q
  double* se = sq + MP;                // MP: e
  double* vm = se + MP;                // KT*MP: mean
  double* saq = vm + KT * MP;          // NAQ: the step's A, Q
  const int M = dm.M, D = dm.D, tid0 = threadIdx.x;
  int tid = tid0, l = tid & 63;
  const int w0 = __builtin_amdgcn_readfirstlane(tid >> 6);
  int w = w0;
  const int k = blockIdx.x;
  typename C::Cov P;
  {  // P0 = Pinf (x) I, m0 = 0
    Model<KT, 0> mdl;
    mdl.init(hy.ls_t[k * hy.stride], hy.var_t[k * hy.stride], 1.0, 1.0);
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      int i, j;
      const bool held = C::position(w, n, i, j);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int gi = 16 * i + (l >> 4) + 4 * q, gj = 16 * j + (l & 15);
        const bool on = gi == gj && gi < M && held;
#pragma unroll
        for (int a = 0; a < KT; ++a)
#pragma unroll
          for (int b = 0; b < KT; ++b) P[n][a][b][q] = on ? mdl.Pinf[a][b] : 0.0;
      }
    }
  }
  for (int e = tid; e < KT * MP; e += NT) vm[e] = 0.0;
  for (int e = tid; e < 16 * kDiagLd; e += NT) sG[e] = 0.0;
  const int64_t k0 = (int64_t)k * dm.T;
  // the next step's L, z and transition are loaded a whole step ahead, before this step's
  // stores: vector memory operations complete in order, so a load behind the packed
  // covariance's stores would wait for them
  double lreg[NL], zreg = 0.0, aqreg = 0.0;
  auto fetch = [&](int64_t kt) {
    const double* L = io.Lw + kt * M * M;
#pragma unroll
    for (int n = 0; n < NL; ++n) {
      const int e = tid + n * NT, r = e / MP, c = e % MP;
      lreg[n] = L[r < M && c < M ? r * M + c : 0];  // masked when it is placed: nothing here waits for the load
    }
    if (tid < M) zreg = io.zw[kt * M + tid];
    if (tid < NAQ) aqreg = io.aq[kt * NAQ + tid];
  };
  auto place = [&]() {
#pragma unroll
    for (int n = 0; n < NL; ++n) {
      const int e = tid + n * NT, r = e / MP, c = e % MP;
      if (NL * NT == MP * MP || e < MP * MP) LT[c * LD + r] = r < M && c < M ? lreg[n] : 0.0;
    }
    if (tid < MP) sq[tid] = zreg;
    if (tid < NAQ) saq[tid] = aqreg;
  };
  auto phase = [&]() { w = fresh_s(w0); tid = fresh_v(tid0); l = tid & 63; };
  fetch(k0);
  place();
  __syncthreads();
#pragma unroll 1
  for (int t = 0; t < dm.T; ++t) {
    phase();
    const int64_t kt = k0 + t;
    double A[KT][KT], Q[KT][KT];
#pragma unroll
    for (int a = 0; a < KT; ++a)
#pragma unroll
      for (int b = 0; b < KT; ++b) {
        A[a][b] = saq[a * KT + b];
        Q[a][b] = saq[KT * KT + a * KT + b];
      }
    C::predict(P, A, Q, M, w, l);
    C::publish(P, X, w, l);
    if (tid < MP) {
      double x[KT];
#pragma unroll
      for (int a = 0; a < KT; ++a) x[a] = vm[a * MP + tid];
#pragma unroll
      for (int a = 0; a < KT; ++a) {
        double v = 0.0;
#pragma unroll
        for (int b = 0; b < KT; ++b) v = fma(A[a][b], x[b], v);
        vm[a * MP + tid] = v;
      }
    }
    __syncthreads();
    phase();
    if (t + 1 < dm.T) fetch(kt + 1);
    // U (row tile w) = P-[:, :M] L: L is lower triangular, column tile j needs inner tiles >= j
    tile4 U[MB];
#pragma unroll
    for (int j = 0; j < MB; ++j) U[j] = tile_zero();
    if (kAllR || w < NR) {
#pragma unroll
      for (int kk = 0; kk < MB; ++kk) {
#pragma unroll
        for (int c = 0; c < 16; c += 4) {
          const double a = frag(X, LD, 16 * w, 16 * kk + c, l);
#pragma unroll
          for (int j = 0; j <= kk; ++j) U[j] = mfma16(a, frag(LT, LD, 16 * j, 16 * kk + c, l), U[j]);
        }
      }
      wave_sync();
#pragma unroll
      for (int j = 0; j < MB; ++j) tile_store(X, LD, 16 * w, 16 * j, U[j], l);
    }
    if (w >= MB) {  // q = z - L' H m-, 16 rows a wavefront
      const int r0 = 16 * (w - MB);
      double v = 0.0;
#pragma unroll
      for (int c = 0; c < MP; c += 4) v = fma(frag(LT, LD, r0, c, l), vm[c + (l >> 4)], v);
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      if (l < 16) sq[r0 + l] -= v;
    }
    __syncthreads();
    phase();
    // the wavefront's second row tile V: row tile w of Mm (w < MB), or q' (the last wavefront)
    tile4 V[MB];
    double quad = 0.0;  // lanes 0-15 of the last wavefront: e' e
    if (w == 0) {
      filter_mm_row<MB, 0>(LT, X, LD, V, l);
      tile_store(sI, kDiagLd, 0, 0, V[0], l);
      wave_sync();
      chol16_inverse(sI, kDiagLd, l);
    } else if (MB > 1 && w == 1) {
      filter_mm_row<MB, (MB > 1 ? 1 : 0)>(LT, X, LD, V, l);
    } else if (MB > 2 && w == 2) {
      filter_mm_row<MB, (MB > 2 ? 2 : 0)>(LT, X, LD, V, l);
    } else if (MB > 3 && w == 3) {
      filter_mm_row<MB, (MB > 3 ? 3 : 0)>(LT, X, LD, V, l);
    } else if (w == NW - 1) {
#pragma unroll
      for (int j = 0; j < MB; ++j) {
        V[j] = tile_zero();
        V[j][0] = l < 16 ? sq[16 * j + l] : 0.0;
      }
    }
    C::template eliminate<true>(P, U, V, quad, X, Lm, sI, sG, se, w0, tid0);
    phase();
    if (t + 1 < dm.T) place();  // LT, sq and saq are not read again in this step
    // m = m- + W e, rows 16 w .. (each wavefront its own)
    if (kAllR || w < NR) {
      double v = 0.0;
#pragma unroll
      for (int c = 0; c < MP; c += 4) v = fma(frag(X, LD, 16 * w, c, l), se[c + (l >> 4)], v);
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      if (l < 16) {
        const double m = vm[16 * w + l] + v;
        vm[16 * w + l] = m;
        const int a = w / MB, i = 16 * (w % MB) + l;
        if (i < M) io.fmean[kt * D + a * M + i] = m;
      }
    }
    if (w == NW - 1) {
      // 1 / sqrt(det Mm): the product of the inverse factors' diagonals
      double m = 1.0;
      int x = 0;
      if (l < MP) m = frexp(sI[(l >> 4) * 16 * kDiagLd + (l & 15) * (kDiagLd + 1)], &x);
      quad = l < 16 ? quad : 0.0;
      for (int o = 32; o > 0; o >>= 1) {
        m *= __shfl_xor(m, o, 64);
        x += __shfl_xor(x, o, 64);
        quad += __shfl_xor(quad, o, 64);
      }
      if (l == 0) {
        io.ell[kt] = quad;
        io.det[2 * kt] = m;
        io.det[2 * kt + 1] = x;
      }
    }
    double* fc = io.fcov + kt * ((int64_t)D * (D + 1) / 2);
    phase();
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      int i, j;
      if (!C::position(w, n, i, j)) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int gi = 16 * i + (l >> 4) + 4 * q, gj = 16 * j + (l & 15);
        if (gi < M && gj < M) {
#pragma unroll
          for (int a = 0; a < KT; ++a) {
            const int r = a * M + gi;
            double* o = fc + r * D - r * (r - 1) / 2 - r + gj;
#pragma unroll
            for (int d = a; d < KT; ++d)
              if (d > a || gi <= gj) o[d * M] = P[n][a][d][q];
          }
          if (KT > 1 && i != j) fc[gj * D - gj * (gj - 1) / 2 - gj + M + gi] = P[n][KT - 1][0][q];
        }
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// RTS backward pass (ops.py:288-311).  The step from t + 1 to t is the affine map
//   m_s = c_t + G_t m_s',  P_s = R_t + G_t P_s' G_t',
//   G_t = P_t A' (P-)^-1,  c_t = m_t - G_t m-,  R_t = P_t - G_t P- G_t'  (P-, m-, A of t + 1),
// whose coefficients depend on the filter only:
//   k_st_gains     the maps of a block of steps of every run, one workgroup per (step, run):
//                  P- = Lc Lc', W = P_t A' Lc^-T, R = P_t - W W', G = W Lc^-1
//   k_st_chain     with few runs, the product of the G_t of a chunk of steps, and
//   k_st_smoother  in COMPOSE mode the chunk's c and R, which make the chunk one map; in JOIN
//                  mode the chunks' maps applied one after the other to the state at the
//                  block's end; in WALK mode every chunk's steps from its right end, with the
//                  outputs H m_s, H P_s H' (the first M states) and, for prediction, the state,
//                  its covariance and the neighbours' cross covariance G_t P_s,t+1.
// One workgroup walks a chunk, so a block of n steps costs n / chunks (compose) + chunks (join)
// + n / chunks (walk) steps instead of n; smoother_chunks() picks the number.
// State layout of these kernels: each of the KT components padded to MP = 16 MB entries, as
// NR = KT MB tiles a side; symmetric matrices as the NR (NR + 1) / 2 tiles (r, j <= r).
// ---------------------------------------------------------------------------
template <int KT, int MB>
struct StTiles {
  static constexpr int MP = 16 * MB, NR = KT * MB, DP = 16 * NR, LD = DP + 2, NF = DP / 4;
  static constexpr int SYM = NR * (NR + 1) / 2 * 256;   // symmetric matrix
  static constexpr int STATE = SYM + DP;                // covariance, mean
  static constexpr int REC = DP * DP + SYM + DP;        // map: G (fragments by row tile), R, c
  static constexpr int SMEM = DP * LD + DP * kDiagLd + 2 * DP;
  // row tile of a wavefront: with eight, wavefronts w and w + 4 share a SIMD, and rows w and 7 - w
  // together have the same number of tiles of a symmetric matrix for every w
  static __device__ int row(int w) { return NR == 8 && w >= 4 ? 11 - w : w; }
  static __device__ int sym(int r, int j) { return (r * (r + 1) / 2 + j) * 256; }
};

struct StGainIO {
  const double* aq;     // [K,T,2 KT^2]
  const double* fmean;  // [K,T,D]
  const double* fcov;   // [K,T,D(D+1)/2]
  double* rec;          // [K, tb] maps
  int t0, tb;
  // STEADY: one map a run, from the filtered covariance fcov [K,D,D] and P- = X [K,D,D] as it stands,
  // aq [K,2 KT^2]; G [K,D,D] is also written as it is
  const double* X;
  double* G;
};

// Per workgroup: 36 + 64 tiles in registers, Lc in LDS.  Bound by the eight pivot chains
// (chol16_inverse) and, behind them, by the matrix instructions of the elimination and of the
// back substitution.  M = 64, D = 128: 999 steps in 293 us (617 us with the sweep inverse of P-
// in LDS and a product through panels).
template <int KT, int MB, bool STEADY>
__global__ __launch_bounds__(64 * KT * MB, 2) void k_st_gains(StDims dm, StGainIO io) {
  using S = StTiles<KT, MB>;
  constexpr int MP = S::MP, NR = S::NR, DP = S::DP, LD = S::LD, NW = NR;
  extern __shared__ double smem[];
  double* X = smem;              // DP x LD: P_t, then Lc (inverse factors on the diagonal tiles)
  double* sW = X + DP * LD;      // DP x kDiagLd: column block b of W; 16 rows of it a wavefront's staging
  double* vp = sW + DP * kDiagLd;  // DP: m-
  const int M = dm.M, D = dm.D, tid = threadIdx.x;
  int l = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), r = S::row(w);
  const int k = blockIdx.y, t = io.t0 + blockIdx.x;
  const int64_t kt = (int64_t)k * dm.T + t, DD = (int64_t)D * D;
  const double* aq = io.aq + (STEADY ? k : kt + 1) * 2 * KT * KT;
  double A[KT][KT], Q[KT][KT];
#pragma unroll
  for (int a = 0; a < KT; ++a)
#pragma unroll
    for (int b = 0; b < KT; ++b) {
      A[a][b] = aq[a * KT + b];
      Q[a][b] = aq[KT * KT + a * KT + b];
    }
  if (STEADY) {  // the filtered covariance, zero padding
    const double* cov = io.fcov + k * DD;
#pragma unroll 4
    for (int pr = w; pr < DP; pr += NW) {
      const int i = pr % MP;
#pragma unroll
      for (int n = 0; n < (DP + 63) / 64; ++n) {
        const int pc = l + 64 * n, j = pc % MP;
        const bool on = i < M && j < M;
        if (pc < DP) X[pr * LD + pc] = on ? cov[(int64_t)(pr / MP * M + i) * D + pc / MP * M + j] : 0.0;
      }
    }
  } else {  // P_t into LDS, both triangles, zero padding
    const double* pk = io.fcov + kt * ((int64_t)D * (D + 1) / 2);
#pragma unroll 4
    for (int pr = w; pr < DP; pr += NW) {
      const int a = pr / MP, i = pr % MP, u = a * M + i;
      const double* row = pk + u * D - u * (u - 1) / 2 - u;
#pragma unroll
      for (int n = 0; n < (DP + 63) / 64; ++n) {
        const int pc = l + 64 * n, b = pc / MP, j = pc % MP;
        if (pc >= pr && pc < DP) {
          const bool on = i < M && j < M;
          const double v = on ? row[b * M + j] : 0.0;
          X[pr * LD + pc] = v;
          X[pc * LD + pr] = v;
        }
      }
    }
    for (int e = tid; e < DP; e += 64 * NW) {
      const int a = e / MP, i = e % MP;
      double v = 0.0;
      if (i < M) {
#pragma unroll
        for (int b = 0; b < KT; ++b) v = fma(aq[a * KT + b], io.fmean[kt * D + b * M + i], v);
      }
      vp[e] = v;
    }
  }
  __syncthreads();
  // row tile r of P- (tiles <= r; identity padding), of P_t A' and of P_t
  tile4 Sm[NR], U[NR], R[NR];
  {
    const int ra = r / MB, ri = r % MB;
    double Ar[KT], Qr[KT];
#pragma unroll
    for (int b = 0; b < KT; ++b) {
      Ar[b] = ra == 0 ? A[0][b] : A[KT - 1][b];
      Qr[b] = ra == 0 ? Q[0][b] : Q[KT - 1][b];
    }
#pragma unroll
    for (int jj = 0; jj < MB; ++jj)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int gi = 16 * ri + (l >> 4) + 4 * q, gj = 16 * jj + (l & 15);
        double own[KT], ap[KT];
#pragma unroll
        for (int b = 0; b < KT; ++b) {
          double p[KT];
#pragma unroll
          for (int a = 0; a < KT; ++a) p[a] = X[(a * MP + gi) * LD + b * MP + gj];
          own[b] = ra == 0 ? p[0] : p[KT - 1];
          ap[b] = 0.0;
#pragma unroll
          for (int a = 0; a < KT; ++a) ap[b] = fma(Ar[a], p[a], ap[b]);
        }
#pragma unroll
        for (int b = 0; b < KT; ++b) {
          double s = gi != gj ? 0.0 : gi < M ? Qr[b] : ra == b ? 1.0 : 0.0, u = 0.0;
#pragma unroll
          for (int a = 0; a < KT; ++a) {
            s = fma(ap[a], A[b][a], s);
            u = fma(own[a], A[b][a], u);
          }
          if (STEADY && gi < M && gj < M) s = io.X[k * DD + (int64_t)(ra * M + gi) * D + b * M + gj];
          Sm[b * MB + jj][q] = s;
          U[b * MB + jj][q] = u;
          R[b * MB + jj][q] = own[b];
        }
      }
  }
  __syncthreads();  // X becomes Lc
  double* st = sW + r * 16 * kDiagLd;
  if (r == 0) {
    tile_store(X, LD, 0, 0, Sm[0], l);
    wave_sync();
    chol16_inverse(X, LD, l);
  }
#pragma unroll
  for (int b = 0; b < NR; ++b) {
    const double* Ib = X + 16 * b * LD + 16 * b;
    __syncthreads();  // inverse factor of diagonal block b
    l = fresh_v(l);
    if (r > b) {
      tile_store(st, kDiagLd, 0, 0, Sm[b], l);
      wave_sync();
      const tile4 v = tile_mul_t(st, kDiagLd, 0, Ib, LD, 0, 0, 0, tile_zero(), l);
      tile_store(X, LD, 16 * r, 16 * b, v, l);
      wave_sync();
    }
    tile_store(st, kDiagLd, 0, 0, U[b], l);
    wave_sync();
    U[b] = tile_mul_t(st, kDiagLd, 0, Ib, LD, 0, 0, 0, tile_zero(), l);
    wave_sync();
    tile_store(st, kDiagLd, 0, 0, U[b], l);
    if (b + 1 < NR && r == b + 1) {  // the next diagonal block first
      double a[4];
      frag4(a, X, LD, 16 * r, 16 * b, 1.0, l);
#pragma unroll
      for (int c = 0; c < 4; ++c) Sm[b + 1] = mfma16(-a[c], a[c], Sm[b + 1]);
      tile_store(X, LD, 16 * r, 16 * r, Sm[b + 1], l);
    }
    __syncthreads();  // column block b of Lc and W
    l = fresh_v(l);
    double a[4];
    if (b + 1 < NR) {
      if (r == b + 1) {
        chol16_inverse(X + 16 * r * LD + 16 * r, LD, l);
      } else if (r > b + 1) {
        frag4(a, X, LD, 16 * r, 16 * b, -1.0, l);
#pragma unroll
        for (int j = b + 1; j < NR; ++j)
          if (j <= r) {
#pragma unroll
            for (int c = 0; c < 4; ++c) Sm[j] = mfma16(a[c], frag(X, LD, 16 * j, 16 * b + 4 * c, l), Sm[j]);
          }
      }
    }
    frag4(a, st, kDiagLd, 0, 0, -1.0, l);
#pragma unroll
    for (int j = b + 1; j < NR; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) U[j] = mfma16(a[c], frag(X, LD, 16 * j, 16 * b + 4 * c, l), U[j]);
#pragma unroll
    for (int j = 0; j < NR; ++j)
      if (j <= r) {
#pragma unroll
        for (int c = 0; c < 4; ++c) R[j] = mfma16(a[c], frag(sW, kDiagLd, 16 * j, 4 * c, l), R[j]);
      }
  }
  double* rec = io.rec + ((int64_t)k * io.tb + blockIdx.x) * S::REC;
#pragma unroll
  for (int j = 0; j < NR; ++j)
    if (j <= r) tile_put(rec + DP * DP + S::sym(r, j), R[j], l);
  __syncthreads();  // every wavefront has read the last column block of W
  // G = W Lc^-1, columns from the last; the rows are the wavefront's own
  double cv = 0.0;
  double* g = rec + r * 16 * DP;
#pragma unroll
  for (int b = NR - 1; b >= 0; --b) {
    l = fresh_v(l);
    double a[4];
    tile_store(st, kDiagLd, 0, 0, U[b], l);
    wave_sync();
    frag4(a, st, kDiagLd, 0, 0, 1.0, l);
    tile4 v = tile_zero();
#pragma unroll
    for (int c = 0; c < 4; ++c) v = mfma16(a[c], frag_t(X, LD, 16 * b + 4 * c, 16 * b, l), v);
    wave_sync();
    tile_store(st, kDiagLd, 0, 0, v, l);
    wave_sync();
    frag4(a, st, kDiagLd, 0, 0, 1.0, l);
    if (STEADY) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int gi = 16 * (r % MB) + (l >> 4) + 4 * q, gj = 16 * (b % MB) + (l & 15);
        if (gi < M && gj < M) io.G[k * DD + (int64_t)(r / MB * M + gi) * D + b / MB * M + gj] = v[q];
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      g[(4 * b + c) * 64 + l] = a[c];
      if (!STEADY) cv = fma(a[c], vp[16 * b + 4 * c + (l >> 4)], cv);
      a[c] = -a[c];
    }
#pragma unroll
    for (int j = 0; j < b; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) U[j] = mfma16(a[c], frag_t(X, LD, 16 * b + 4 * c, 16 * j, l), U[j]);
    wave_sync();
  }
  if (STEADY) return;
  cv += __shfl_xor(cv, 16, 64);
  cv += __shfl_xor(cv, 32, 64);
  if (l < 16) {
    const int i = 16 * (r % MB) + l;
    rec[DP * DP + S::SYM + 16 * r + l] = i < M ? io.fmean[kt * D + (r / MB) * M + i] - cv : 0.0;
  }
}

struct StSmootherIO {
  double* rec;       // [K, tb] maps of the block's steps
  double* comp;      // [K, nc] maps of its chunks
  double* state;     // [K, slots] states: 0 / 1 the block's right end and its result, 2 + c the right
                     // end of chunk c
  int tb, nc, slots, in;  // in: slot of the right end (0 or 1)
  int t0, nb;        // the block's first step, its number of steps
  double* pm;        // [K,T,M]
  double* pP;        // [K,T,M,M]
  double* smean;     // optional [K,T,D] smoothed state (return_full)
  double* scov;      // optional [K,T,D,D]
  double* scross;    // optional [K,T,D,D]: G_t P_s,t+1 = Cov(x_t, x_t+1 | y); Pinf at the last step
  double* xs;        // ST_STEADY: [K,D,D] in and out
  int iters;
};

// first step of chunk c of a block
__device__ inline int chunk_start(const StSmootherIO& io, int c) { return (int)((int64_t)io.nb * c / io.nc); }

// The last step: the smoothed state is the filtered one (ops.py:314-315).
template <int KT, int MB>
__global__ __launch_bounds__(kT) void k_st_terminal(StDims dm, StHyp hy, const double* __restrict__ fmean,
                                                    const double* __restrict__ fcov, StSmootherIO io) {
  using S = StTiles<KT, MB>;
  const int M = dm.M, D = dm.D, tid = threadIdx.x, k = blockIdx.x;
  const int64_t kt = (int64_t)k * dm.T + dm.T - 1, DD = (int64_t)D * D;
  const double* pk = fcov + kt * ((int64_t)D * (D + 1) / 2);
  double* st = io.state + (int64_t)k * io.slots * S::STATE;
  for (int e = tid; e < S::SYM; e += kT) {
    int tile = e >> 8, r = 0;
    while (tile > r) tile -= ++r;
    const int l = (e & 255) >> 2, q = e & 3;
    const int pi = 16 * r + (l >> 4) + 4 * q, pj = 16 * tile + (l & 15);
    const int i = pi % S::MP, j = pj % S::MP, u = pi / S::MP * M + i, v = pj / S::MP * M + j;
    st[e] = (i < M && j < M) ? pk[u <= v ? pidx(u, v, D) : pidx(v, u, D)] : 0.0;
  }
  for (int e = tid; e < S::DP; e += kT) {
    const int i = e % S::MP;
    st[S::SYM + e] = i < M ? fmean[kt * D + e / S::MP * M + i] : 0.0;
  }
  for (int e = tid; e < M; e += kT) io.pm[kt * M + e] = fmean[kt * D + e];
  for (int e = tid; e < M * M; e += kT) {
    const int i = e / M, j = e % M;
    io.pP[kt * M * M + e] = pk[i <= j ? pidx(i, j, D) : pidx(j, i, D)];
  }
  if (io.smean) {
    Model<KT, 0> mdl;
    mdl.init(hy.ls_t[k * hy.stride], hy.var_t[k * hy.stride], 1.0, 1.0);
    for (int e = tid; e < D; e += kT) io.smean[kt * D + e] = fmean[kt * D + e];
    for (int64_t e = tid; e < DD; e += kT) {
      const int i = (int)(e / D), j = (int)(e % D);
      io.scov[kt * DD + e] = pk[i <= j ? pidx(i, j, D) : pidx(j, i, D)];
      io.scross[kt * DD + e] = (i % M == j % M) ? mdl.Pinf[i / M][j / M] : 0.0;
    }
  }
}

// Product of the G_t of chunk blockIdx.x + 1, block per (chunk, run): E = G_first ... G_last,
// from the last factor, with E' in LDS.
template <int KT, int MB>
__global__ __launch_bounds__(64 * KT * MB, 2) void k_st_chain(StSmootherIO io) {
  using S = StTiles<KT, MB>;
  constexpr int NR = S::NR, DP = S::DP, LD = S::LD, NF = S::NF;
  extern __shared__ double X[];  // DP x LD: E'
  const int l = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = blockIdx.x + 1, k = blockIdx.y;
  const int s0 = chunk_start(io, c), s1 = chunk_start(io, c + 1);
  const double* src = io.rec + (int64_t)k * io.tb * S::REC + w * 16 * DP + l;
  double g[NF];
  auto fetch = [&](int s) {
#pragma unroll
    for (int f = 0; f < NF; ++f) g[f] = src[(int64_t)s * S::REC + f * 64];
  };
  fetch(s1 - 1);
#pragma unroll
  for (int f = 0; f < NF; ++f) X[(4 * f + (l >> 4)) * LD + 16 * w + (l & 15)] = g[f];
#pragma unroll 1
  for (int s = s1 - 2; s >= s0; --s) {
    fetch(s);
    __syncthreads();
    tile4 E[NR];
#pragma unroll
    for (int j = 0; j < NR; ++j) E[j] = tile_zero();
#pragma unroll
    for (int f = 0; f < NF; ++f) {
#pragma unroll
      for (int j = 0; j < NR; ++j) E[j] = mfma16(g[f], frag(X, LD, 16 * j, 4 * f, l), E[j]);
      if (f % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NR; ++j) tile_store_t(X, LD, 16 * j, 16 * w, E[j], l);
  }
  __syncthreads();
  double* out = io.comp + ((int64_t)k * io.nc + c) * S::REC + w * 16 * DP + l;
#pragma unroll
  for (int f = 0; f < NF; ++f) out[f * 64] = frag_t(X, LD, 4 * f, 16 * w, l);
}

// ST_STEADY: `iters` times the run's one map, on the covariance xs (the infinite-horizon smoother).
enum { ST_WALK = 0, ST_COMPOSE = 1, ST_JOIN = 2, ST_STEADY = 3 };

// Per step T = G P_s' (G's row tile from registers, P_s' in LDS, both triangles) and
// P_s = R + T G' (tiles j <= r; G in LDS, T through a staging tile): 51 k cycles of FP64 matrix
// instructions a SIMD at D = 128, which bound it; the next step's G is on its way meanwhile.
// 28 us a step, 35 with the outputs (89 us with both products through LDS panels of 8 columns);
// one run of 1000 steps in 45 chunks: 3.3 ms for the whole pass (89 ms for those products walked
// as one chain).
template <int KT, int MB, int MODE>
__global__ __launch_bounds__(64 * KT * MB, 2) void k_st_smoother(StDims dm, StSmootherIO io) {
  using S = StTiles<KT, MB>;
  constexpr int MP = S::MP, NR = S::NR, DP = S::DP, LD = S::LD, NF = S::NF, NT = 64 * NR;
  extern __shared__ double smem[];
  double* X = smem;                  // DP x LD: P_s', then G
  double* sT = X + DP * LD;          // NR of 16 x kDiagLd: staging tiles
  double* ms = sT + DP * kDiagLd;    // 2 x DP: means, alternating
  const int M = dm.M, D = dm.D, tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), r = S::row(w);
  int l = tid & 63;
  const int k = blockIdx.y;
  const int c = MODE == ST_COMPOSE ? blockIdx.x + 1 : blockIdx.x;
  const int s0 = MODE == ST_STEADY ? 0 : MODE == ST_JOIN ? 1 : chunk_start(io, c);
  const int s1 = MODE == ST_STEADY ? io.iters : MODE == ST_JOIN ? io.nc : chunk_start(io, c + 1);
  const double* rec = MODE == ST_JOIN ? io.comp + (int64_t)k * io.nc * S::REC : io.rec + (int64_t)k * io.tb * S::REC;
  double* states = io.state + (int64_t)k * io.slots * S::STATE;
  double* st = sT + w * 16 * kDiagLd;
  tile4 P[NR];
  if (MODE == ST_STEADY) {
    const double* xs = io.xs + (int64_t)k * D * D;
#pragma unroll
    for (int j = 0; j < NR; ++j)
      if (j <= r) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int gi = 16 * (r % MB) + (l >> 4) + 4 * q, gj = 16 * (j % MB) + (l & 15);
          P[j][q] = gi < M && gj < M ? xs[(int64_t)(r / MB * M + gi) * D + j / MB * M + gj] : 0.0;
        }
      }
    for (int e = tid; e < DP; e += NT) ms[e] = 0.0;
  } else if (MODE == ST_COMPOSE) {
#pragma unroll
    for (int j = 0; j < NR; ++j) P[j] = tile_zero();
    for (int e = tid; e < DP; e += NT) ms[e] = 0.0;
  } else {
    const double* in = states + (MODE == ST_WALK && c + 1 < io.nc ? 2 + c : io.in) * S::STATE;
#pragma unroll
    for (int j = 0; j < NR; ++j)
      if (j <= r) P[j] = tile_get(in + S::sym(r, j), l);
    for (int e = tid; e < DP; e += NT) ms[e] = in[S::SYM + e];
  }
  double g[NF];
  auto fetch = [&](int s) {
    const double* src = rec + (MODE == ST_STEADY ? 0 : (int64_t)s * S::REC) + r * 16 * DP + l;
#pragma unroll
    for (int f = 0; f < NF; ++f) g[f] = src[f * 64];
  };
  auto publish = [&]() {  // P_s into LDS, both triangles
#pragma unroll
    for (int j = 0; j < NR; ++j)
      if (j <= r) {
        tile_store(X, LD, 16 * r, 16 * j, P[j], l);
        if (j != r) tile_store_t(X, LD, 16 * j, 16 * r, P[j], l);
      }
  };
  auto emit = [&](int s, const double* mean) {  // outputs of step s from LDS
    const int64_t kt = (int64_t)k * dm.T + io.t0 + s;
    for (int e = tid; e < M; e += NT) io.pm[kt * M + e] = mean[e];
    for (int e = tid; e < M * M; e += NT) io.pP[kt * M * M + e] = X[(e / M) * LD + e % M];
    if (io.smean) {
      for (int e = tid; e < D; e += NT) io.smean[kt * D + e] = mean[e / M * MP + e % M];
      for (int e = tid; e < D * D; e += NT) {
        const int i = e / D, j = e % D;
        io.scov[kt * D * D + e] = X[(i / M * MP + i % M) * LD + j / M * MP + j % M];
      }
    }
  };
  if (s0 < s1) fetch(s1 - 1);
  int cur = 0;
#pragma unroll 1
  for (int s = s1 - 1; s >= s0; --s) {
    l = fresh_v(l);
    publish();
    __syncthreads();
    if (MODE == ST_WALK && s + 1 < s1) emit(s + 1, ms + cur * DP);
    const double* rs = rec + (MODE == ST_STEADY ? 0 : (int64_t)s * S::REC) + DP * DP;
    tile4 T[NR];
    double v = 0.0;
#pragma unroll
    for (int j = 0; j < NR; ++j) T[j] = tile_zero();
#pragma unroll
    for (int f = 0; f < NF; ++f) {
#pragma unroll
      for (int j = 0; j < NR; ++j) T[j] = mfma16(g[f], frag(X, LD, 16 * j, 4 * f, l), T[j]);
      if (MODE != ST_STEADY) v = fma(g[f], ms[cur * DP + 4 * f + (l >> 4)], v);
      if (f % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    }
    if (MODE != ST_STEADY) {
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      cur ^= 1;
      if (l < 16) ms[cur * DP + 16 * r + l] = rs[S::SYM + 16 * r + l] + v;
    }
    if (MODE == ST_WALK && io.scross) {
      const int64_t kt = (int64_t)k * dm.T + io.t0 + s;
#pragma unroll
      for (int j = 0; j < NR; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int gi = 16 * (r % MB) + (l >> 4) + 4 * q, gj = 16 * (j % MB) + (l & 15);
          if (gi < M && gj < M) io.scross[kt * D * D + (int64_t)(r / MB * M + gi) * D + j / MB * M + gj] = T[j][q];
        }
    }
#pragma unroll
    for (int j = 0; j < NR; ++j)
      if (j <= r) P[j] = tile_get(rs + S::sym(r, j), l);
    __syncthreads();  // P_s' is read
#pragma unroll
    for (int f = 0; f < NF; ++f) X[(16 * r + (l & 15)) * LD + 4 * f + (l >> 4)] = g[f];
    __syncthreads();  // G
    l = fresh_v(l);
    if (s > s0) fetch(s - 1);
#pragma unroll
    for (int b = 0; b < NR; ++b) {
      double a[4];
      tile_store(st, kDiagLd, 0, 0, T[b], l);
      wave_sync();
      frag4(a, st, kDiagLd, 0, 0, 1.0, l);
      wave_sync();
#pragma unroll
      for (int j = 0; j < NR; ++j)
        if (j <= r) {
#pragma unroll
          for (int e = 0; e < 4; ++e) P[j] = mfma16(a[e], frag(X, LD, 16 * j, 16 * b + 4 * e, l), P[j]);
        }
    }
    __syncthreads();  // G is read
    if (MODE == ST_JOIN) {  // the right end of chunk s - 1
      double* o = states + (2 + s - 1) * S::STATE;
#pragma unroll
      for (int j = 0; j < NR; ++j)
        if (j <= r) tile_put(o + S::sym(r, j), P[j], l);
      for (int e = tid; e < DP; e += NT) o[S::SYM + e] = ms[cur * DP + e];
    }
  }
  if (MODE == ST_STEADY) {
    double* xs = io.xs + (int64_t)k * D * D;
#pragma unroll
    for (int j = 0; j < NR; ++j)
      if (j <= r) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int gi = 16 * (r % MB) + (l >> 4) + 4 * q, gj = 16 * (j % MB) + (l & 15);
          const int u = r / MB * M + gi, v = j / MB * M + gj;
          if (gi < M && gj < M) {
            xs[(int64_t)u * D + v] = P[j][q];
            if (j != r) xs[(int64_t)v * D + u] = P[j][q];
          }
        }
      }
  }
  if (MODE == ST_WALK) {
    publish();
    __syncthreads();
    if (s0 < s1) emit(s0, ms + cur * DP);
  }
  if (MODE == ST_COMPOSE || (MODE == ST_WALK && c == 0)) {
    double* o = MODE == ST_COMPOSE ? io.comp + ((int64_t)k * io.nc + c) * S::REC + DP * DP
                                   : states + (1 - io.in) * S::STATE;
#pragma unroll
    for (int j = 0; j < NR; ++j)
      if (j <= r) tile_put(o + S::sym(r, j), P[j], l);
    for (int e = tid; e < DP; e += NT) o[S::SYM + e] = ms[cur * DP + e];
  }
}

// bytes of the block of maps: 2500 steps of one d = 128 run, 12 steps each of 200 runs
constexpr int64_t kGainBudget = int64_t(512) << 20;
// Workgroups that run side by side: one a compute unit (k_st_smoother fills a unit's LDS).
constexpr int kUnits = 256;

// doubles of one map / one state of the smoother (StTiles::REC, STATE)
int64_t map_doubles(const StDims& dm) {
  const int64_t nr = dm.KT * ((dm.M + 15) / 16), dp = 16 * nr;
  return dp * dp + nr * (nr + 1) / 2 * 256 + dp;
}
int64_t state_doubles(const StDims& dm) {
  const int64_t nr = dm.KT * ((dm.M + 15) / 16);
  return nr * (nr + 1) / 2 * 256 + 16 * nr;
}

int gain_block_steps(const StDims& dm) {
  const int64_t per = (int64_t)dm.K * map_doubles(dm) * (int64_t)sizeof(double);
  int64_t tb = kGainBudget / per;
  const int64_t need = dm.T > 1 ? dm.T - 1 : 1;
  if (tb > need) tb = need;
  if (tb < 1) tb = 1;
  return (int)tb;
}

// Chunks per run of a block of nb steps.  Four launches follow each other: k_st_chain (one
// product a step) and COMPOSE (two) over the steps of a chunk, JOIN over the chunks, WALK over
// the steps again.  2 ceil(nb / c) + c - 1 steps of the walk stand for them, against nb for one
// chunk: at D = 128, 999 steps in 45 chunks, CHAIN and COMPOSE take 18 and 33 us a step, JOIN
// 28 us a chunk, WALK 35 us a step, 3.2 ms in all (as one walk, 35 ms by that rate).  Chunks are taken up to
// half as many as there are units, in all runs together; whether more pay for 32 to 128 runs,
// where each launch then leaves units idle, has not been measured.
int smoother_chunks(const StDims& dm, int nb) {
  int best = 1, cost = nb;
  for (int c = 2; c <= nb && 2 * (int64_t)c * dm.K <= kUnits; ++c) {
    const int n = 2 * ((nb + c - 1) / c) + c - 1;
    if (n < cost) { best = c; cost = n; }
  }
  return best;
}
int smoother_max_chunks(const StDims& dm) {
  const int64_t c = kUnits / (2 * (int64_t)dm.K);
  return c > 1 ? (int)c : 1;
}

// per-run sums of per-step partials: out[k] = sum_t a[k*T + t]
__global__ __launch_bounds__(kT) void k_st_sum(int32_t T, const double* __restrict__ a, double* __restrict__ out) {
  __shared__ double red[4];
  const int k = blockIdx.x;
  double s = 0.0;
  for (int t = threadIdx.x; t < T; t += kT) s += a[(int64_t)k * T + t];
  s = wg_sum(s, red);
  if (threadIdx.x == 0) out[k] = s;
}

// ---------------------------------------------------------------------------
// Mean-field space-time filter and smoother (ops.py:429-706, the filter and smoother of
// MarkovMeanFieldGaussianProcess, basemodels.py:1158-1175).  The state is M independent
// temporal blocks (block i = the KT-dim state of latent i, kernels.py:526-575); each update
// keeps only the diagonal blocks of the state covariance.  With P block diagonal and
// H = I_M (x) e_0', the dense update of ops.py:452-461 reduces to
//   S = R + diag(d),  d_i = P-_i[0][0],  v = y - (m-_i[0])_i,  u = S^-1 v,
//   m_i = m-_i + P-_i e_0 u_i,  P_i = P-_i - [S^-1]_ii (P-_i e_0)(P-_i e_0)'
// (block i of K H P- is P-_i e_0 [S^-1]_ii e_0' P-_i: only the diagonal of S^-1 reaches it).
// The associative-scan form (ops.py:468-578) builds every element from S_t = R_t + diag(h Q_t h')
// and projects it to the blocks; per block its elements are those of an ordinary scalar-
// observation filter with noise r_i = 1/[S_t^-1]_ii - h Q_t,i h' and observation
// [S_t^-1 y_t]_i / [S_t^-1]_ii, which k_mf_blocks runs; its log likelihood is then taken
// from the predictions with the dense S (ops.py:572-576).
// Layouts: y [K,T,M], noise R [K,T,M,M] (symmetric), block means [K,T,M,KT], block
// covariances [K,T,M,KT,KT].
// ---------------------------------------------------------------------------

// Pseudo observation of compute_full_pseudo_lik (basemodels.py:676-687) from the whitened
// form: R = (L L')^-1, y = R L z.  Block per (step, run); L L' on the matrix cores, the
// inverse by the sweep operator in LDS.
__global__ __launch_bounds__(kT) void k_mf_pseudo(StDims dm, const double* __restrict__ Lw,
                                                  const double* __restrict__ zw, double* __restrict__ R,
                                                  double* __restrict__ y) {
  extern __shared__ double smem[];
  double* pan = smem;                 // 2*kPK*kPS
  double* sW = pan + 2 * kPK * kPS;   // M*M
  double* row = sW + kMaxM * kMaxM;   // 2*kMaxM
  double* sv = row + 2 * kMaxM;       // M
  const int t = blockIdx.x, k = blockIdx.y, M = dm.M, tid = threadIdx.x;
  const int64_t kt = (int64_t)k * dm.T + t;
  const double* L = Lw + kt * M * M;  // lower triangular, upper part zero
  wg_gemm_small(M, M, M, 1.0, MatRef{L, M, 1}, MatRef{L, 1, M}, 0.0, sW, M, pan);
  if (tid < M) {
    double s = 0.0;
    for (int q = 0; q <= tid; ++q) s = fma(L[tid * M + q], zw[kt * M + q], s);
    sv[tid] = s;
  }
  wg_sweep_inv<kMaxM / 16, false>(sW, M, M, row);  // sW = -(L L')^-1
  double* Rk = R + kt * M * M;
  for (int e = tid; e < M * M; e += kT) Rk[e] = -sW[e];
  if (tid < M) {
    double s = 0.0;
    for (int j = 0; j < M; ++j) s = fma(-sW[tid * M + j], sv[j], s);
    y[kt * M + tid] = s;
  }
}

struct MfFilterIO {
  const double* dt;   // [K,T] (dt[k,0] = 0 for the first step of a run)
  const double* y;    // [K,T,M]
  const double* R;    // [K,T,M,M]
  double* fmean;      // [K,T,M,KT]
  double* fcov;       // [K,T,M,KT,KT]
  double* ell;        // [K,T]
  double* reff;       // [K,T,M] (associative form)
  double* yeff;       // [K,T,M]
};

template <int KT>
__device__ inline void mf_predict(const double A[KT * KT], const double Q[KT * KT], const double m[KT],
                                  const double P[KT][KT], double mp[KT], double Pp[KT][KT]) {
  double AP[KT][KT];
  for (int i = 0; i < KT; ++i) {
    double s = 0.0;
    for (int q = 0; q < KT; ++q) s = fma(A[i * KT + q], m[q], s);
    mp[i] = s;
    for (int j = 0; j < KT; ++j) {
      double a = 0.0;
      for (int q = 0; q < KT; ++q) a = fma(A[i * KT + q], P[q][j], a);
      AP[i][j] = a;
    }
  }
  for (int i = 0; i < KT; ++i)
    for (int j = 0; j < KT; ++j) {
      double s = Q[i * KT + j];
      for (int q = 0; q < KT; ++q) s = fma(AP[i][q], A[j * KT + q], s);
      Pp[i][j] = s;
    }
  for (int i = 0; i < KT; ++i)
    for (int j = i + 1; j < KT; ++j) Pp[i][j] = Pp[j][i] = 0.5 * (Pp[i][j] + Pp[j][i]);
}

template <int KT>
__device__ inline void mf_pinf(double ls, double var, double P[KT][KT]) {
  Model<KT, 0> mdl;
  mdl.init(ls, var, 1.0, 1.0);
  for (int i = 0; i < KT; ++i)
    for (int j = 0; j < KT; ++j) P[i][j] = mdl.Pinf[i][j];
}

// Sequential form (ops.py:429-465): block per run, loop over T.  Thread i < M owns block i
// in registers; S = R_t + diag(d) is inverted in LDS by the sweep operator (log det from
// its pivots).
template <int KT>
__global__ __launch_bounds__(kT) void k_mf_filter(StDims dm, StHyp hy, MfFilterIO io) {
  __shared__ double sS[kMaxM * kMaxM];
  __shared__ double row[2 * kMaxM];
  __shared__ double sv[kMaxM];
  __shared__ double red[4];
  const int k = blockIdx.x, M = dm.M, tid = threadIdx.x;
  const double ls = hy.ls_t[k * hy.stride], var = hy.var_t[k * hy.stride];
  double m[KT], P[KT][KT], mp[KT], Pp[KT][KT];
  mf_pinf<KT>(ls, var, P);
  for (int i = 0; i < KT; ++i) m[i] = 0.0;
  for (int t = 0; t < dm.T; ++t) {
    const int64_t kt = (int64_t)k * dm.T + t;
    const double* Rt = io.R + kt * M * M;
    for (int e = tid; e < M * M; e += kT) sS[e] = Rt[e];
    if (tid < M) {
      double A[KT * KT], Q[KT * KT];
      temporal_AQ<KT>(ls, var, io.dt[kt], A, Q);
      mf_predict<KT>(A, Q, m, P, mp, Pp);
      sv[tid] = io.y[kt * M + tid] - mp[0];
    }
    __syncthreads();
    if (tid < M) sS[tid * M + tid] += Pp[0][0];
    const double ld = wg_sweep_inv<kMaxM / 16, true>(sS, M, M, row);  // sS = -S^-1
    double q = 0.0, u = 0.0, s = 0.0;
    if (tid < M) {
      for (int j = 0; j < M; ++j) u = fma(-sS[tid * M + j], sv[j], u);
      s = -sS[tid * M + tid];
      q = sv[tid] * u;
    }
    const double quad = wg_sum(q, red);
    if (tid == 0) io.ell[kt] = -0.5 * (quad + M * kLog2Pi + ld);
    if (tid < M) {
      double* fm = io.fmean + (kt * M + tid) * KT;
      double* fc = io.fcov + (kt * M + tid) * KT * KT;
      for (int i = 0; i < KT; ++i) {
        m[i] = fma(Pp[i][0], u, mp[i]);
        fm[i] = m[i];
        for (int j = 0; j < KT; ++j) {
          P[i][j] = fma(-s * Pp[i][0], Pp[j][0], Pp[i][j]);
          fc[i * KT + j] = P[i][j];
        }
      }
    }
  }
}

// Per-step dense part of the associative form, block per (step, run).
//   ELEMENTS: d = h Q_t h' (Q_0 = Pinf), reff_i = 1/[S^-1]_ii - d_i, yeff_i = [S^-1 y]_i / [S^-1]_ii
//   LOGLIK:   d, v from the prediction of the filtered blocks at t-1 (Pinf, 0 at t = 0),
//             ell_t = log N(v | 0, S)
template <int KT, bool LOGLIK>
__global__ __launch_bounds__(kT) void k_mf_sdiag(StDims dm, StHyp hy, MfFilterIO io) {
  __shared__ double sS[kMaxM * kMaxM];
  __shared__ double row[2 * kMaxM];
  __shared__ double sv[kMaxM];
  __shared__ double red[4];
  const int t = blockIdx.x, k = blockIdx.y, M = dm.M, tid = threadIdx.x;
  const int64_t kt = (int64_t)k * dm.T + t;
  const double ls = hy.ls_t[k * hy.stride], var = hy.var_t[k * hy.stride];
  const double* Rt = io.R + kt * M * M;
  for (int e = tid; e < M * M; e += kT) sS[e] = Rt[e];
  double d = 0.0;
  if (tid < M) {
    double P[KT][KT];
    mf_pinf<KT>(ls, var, P);
    double A[KT * KT], Q[KT * KT];
    temporal_AQ<KT>(ls, var, io.dt[kt], A, Q);
    if (!LOGLIK) {
      d = t == 0 ? P[0][0] : Q[0];
      sv[tid] = io.y[kt * M + tid];
    } else {
      double m[KT], mp[KT], Pp[KT][KT];
      for (int i = 0; i < KT; ++i) m[i] = 0.0;
      if (t > 0) {
        const double* fm = io.fmean + ((kt - 1) * M + tid) * KT;
        const double* fc = io.fcov + ((kt - 1) * M + tid) * KT * KT;
        for (int i = 0; i < KT; ++i) {
          m[i] = fm[i];
          for (int j = 0; j < KT; ++j) P[i][j] = fc[i * KT + j];
        }
      }
      mf_predict<KT>(A, Q, m, P, mp, Pp);
      d = Pp[0][0];
      sv[tid] = io.y[kt * M + tid] - mp[0];
    }
  }
  __syncthreads();
  if (tid < M) sS[tid * M + tid] += d;
  const double ld = wg_sweep_inv<kMaxM / 16, LOGLIK>(sS, M, M, row);  // sS = -S^-1
  double q = 0.0, u = 0.0;
  if (tid < M) {
    for (int j = 0; j < M; ++j) u = fma(-sS[tid * M + j], sv[j], u);
    q = sv[tid] * u;
  }
  if (LOGLIK) {
    const double quad = wg_sum(q, red);
    if (tid == 0) io.ell[kt] = -0.5 * (quad + M * kLog2Pi + ld);
  } else if (tid < M) {
    const double s = -sS[tid * M + tid];
    io.reff[kt * M + tid] = 1.0 / s - d;
    io.yeff[kt * M + tid] = u / s;
  }
}

// The recursions over time of the mean-field blocks: one wavefront walks 64 (run, block) pairs
// and is bound by its own chain of dependent FP64 operations, so everything that does not depend
// on the previous step is made by other wavefronts of the workgroup, a tile of steps ahead, and
// handed over in LDS.  Transitions depend on the run and the step alone: the workgroup makes
// them once for each of the runs that its lanes belong to.
constexpr int kMfTile = 8;

// Lanes of a walker: 64, but 32 where the smoother's fields and the transitions of so many runs
// would exceed the LDS.
inline int mf_lanes(const StDims& dm) { return dm.M <= 2 ? 32 : 64; }
inline int mf_runs(const StDims& dm) { return (mf_lanes(dm) + dm.M - 2) / dm.M + 1; }  // most of one walker
inline size_t mf_table_doubles(const StDims& dm) { return (size_t)2 * mf_runs(dm) * kMfTile * 2 * dm.KT * dm.KT; }

// Transitions of the steps first + dir * (0 .. kMfTile - 1) of the runs k0 .. k0 + nr - 1; steps
// outside a run repeat its first or last.
template <int KT>
__device__ void mf_transitions(const StDims& dm, const StHyp& hy, const double* dt, int k0, int nr, int first, int dir,
                               double* aq, int tid, int n) {
  for (int e = tid; e < nr * kMfTile; e += n) {
    const int k = k0 + e / kMfTile;
    const int t = min(max(first + dir * (e % kMfTile), 0), dm.T - 1);
    double A[KT * KT], Q[KT * KT];
    temporal_AQ<KT>(hy.ls_t[k * hy.stride], hy.var_t[k * hy.stride], dt[(int64_t)k * dm.T + t], A, Q);
    double* o = aq + e * 2 * KT * KT;
    for (int j = 0; j < KT * KT; ++j) { o[j] = A[j]; o[KT * KT + j] = Q[j]; }
  }
}

// Scalar-observation filter of every block over the per-step (reff, yeff): wavefront 0 walks, a
// lane per (run, block), two more make the next tile's transitions.  4 runs of 500 steps at
// M = 64: 377 -> 136 us (with the transitions in the walk, and every load waited for
// where it is used).
constexpr int kMfBlocksT = 192;
template <int KT>
__global__ __launch_bounds__(kMfBlocksT) void k_mf_blocks(StDims dm, StHyp hy, MfFilterIO io, int lanes) {
  extern __shared__ double smem[];
  const int M = dm.M, T = dm.T, lane = threadIdx.x & 63;
  const bool walker = threadIdx.x < 64;
  const int64_t total = (int64_t)dm.K * M, g0 = (int64_t)blockIdx.x * lanes;
  const int64_t last = min(g0 + lanes, total) - 1;
  const bool mine = walker && lane < lanes && g0 + lane < total;
  const int64_t g = min(g0 + min(lane, lanes - 1), total - 1);
  const int k0 = (int)(g0 / M), nr = (int)(last / M) - k0 + 1;
  const int k = (int)(g / M), i = (int)(g % M);
  const int table = nr * kMfTile * 2 * KT * KT;
  const int64_t row0 = (int64_t)k * T * M + i;  // of step 0; steps are M apart
  double m[KT], P[KT][KT], r[kMfTile], y[kMfTile];
  mf_pinf<KT>(hy.ls_t[k * hy.stride], hy.var_t[k * hy.stride], P);
  for (int a = 0; a < KT; ++a) m[a] = 0.0;
  if (walker) {
#pragma unroll
    for (int s = 0; s < kMfTile; ++s) {
      const int64_t e = row0 + (int64_t)min(s, T - 1) * M;
      r[s] = io.reff[e];
      y[s] = io.yeff[e];
    }
  } else {
    mf_transitions<KT>(dm, hy, io.dt, k0, nr, 0, 1, smem, threadIdx.x - 64, kMfBlocksT - 64);
  }
  __syncthreads();
  for (int t0 = 0, n = 0; t0 < T; t0 += kMfTile, ++n) {
    if (walker) {
      const double* aq = smem + (n & 1) * table + (k - k0) * kMfTile * 2 * KT * KT;
      double rn[kMfTile], yn[kMfTile];
#pragma unroll
      for (int s = 0; s < kMfTile; ++s) {
        const int64_t e = row0 + (int64_t)min(t0 + kMfTile + s, T - 1) * M;
        rn[s] = io.reff[e];
        yn[s] = io.yeff[e];
      }
#pragma unroll
      for (int s = 0; s < kMfTile; ++s) {
        double mp[KT], Pp[KT][KT], A[KT * KT], Q[KT * KT];
        for (int j = 0; j < KT * KT; ++j) { A[j] = aq[s * 2 * KT * KT + j]; Q[j] = aq[(s * 2 + 1) * KT * KT + j]; }
        mf_predict<KT>(A, Q, m, P, mp, Pp);
        const double S = Pp[0][0] + r[s], v = y[s] - mp[0];
        for (int a = 0; a < KT; ++a) {
          const double Ka = Pp[a][0] / S;
          m[a] = fma(Ka, v, mp[a]);
          for (int b = 0; b < KT; ++b) P[a][b] = fma(-Ka, Pp[b][0], Pp[a][b]);
        }
        if (mine && t0 + s < T) {
          const int64_t e = row0 + (int64_t)(t0 + s) * M;
          for (int a = 0; a < KT; ++a) {
            io.fmean[e * KT + a] = m[a];
            for (int b = 0; b < KT; ++b) io.fcov[(e * KT + a) * KT + b] = P[a][b];
          }
        }
      }
#pragma unroll
      for (int s = 0; s < kMfTile; ++s) { r[s] = rn[s]; y[s] = yn[s]; }
    } else if (t0 + kMfTile < T) {
      mf_transitions<KT>(dm, hy, io.dt, k0, nr, t0 + kMfTile, 1, smem + ((n + 1) & 1) * table, threadIdx.x - 64,
                         kMfBlocksT - 64);
    }
    __syncthreads();
  }
}

struct MfSmootherIO {
  const double* dt;     // [K,T] step vector of the smoother (already the next step's dt)
  const double* fmean;  // [K,T,M,KT]
  const double* fcov;   // [K,T,M,KT,KT]
  double* hmean;        // optional [K,T,M]: h m_s
  double* hvar;         // optional: h P_s h' at hvar[kt*var_step + i*var_elem]
  int64_t var_step, var_elem;
  double* smean;        // optional [K,T,M,KT]
  double* scov;         // optional [K,T,M,KT,KT]
  double* gain;         // optional [K,T,M,KT,KT]
};

// RTS smoother of every block (ops.py:611-641; the associative form 644-678 gives the
// same result), lane per (run, block), from the last step back.  Wavefront 0 walks a tile of
// steps while eight others, a step each, make the next tile's gains and predictions (about 130
// of the 200 operations of a step, its four divisions among them) and after that the transitions
// of the tile after next.  4 runs of 500 steps at M = 64: 310 -> 119 us.
constexpr int kMfSmootherT = 64 * (kMfTile + 1);
template <int KT>
constexpr int kMfFields = 2 * KT + 3 * KT * KT;  // fm, pm, fP, pP, G

template <int KT>
__global__ __launch_bounds__(kMfSmootherT) void k_mf_smoother(StDims dm, StHyp hy, MfSmootherIO io, int lanes) {
  extern __shared__ double smem[];
  constexpr int K2 = KT * KT, F = kMfFields<KT>;
  const int M = dm.M, T = dm.T, lane = threadIdx.x & 63, s_own = (int)(threadIdx.x >> 6) - 1;
  const int64_t total = (int64_t)dm.K * M, g0 = (int64_t)blockIdx.x * lanes;
  const int64_t last = min(g0 + lanes, total) - 1;
  const bool mine = lane < lanes && g0 + lane < total;
  const int64_t g = min(g0 + min(lane, lanes - 1), total - 1);
  const int k0 = (int)(g0 / M), nr = (int)(last / M) - k0 + 1;
  const int k = (int)(g / M), i = (int)(g % M);
  const int table = nr * kMfTile * 2 * K2;
  double* fields = smem;                      // [2][kMfTile][F][64]
  double* aq = smem + 2 * kMfTile * F * 64;   // [2][nr][kMfTile][2 K2]
  const int tiles = (T + kMfTile - 1) / kMfTile;
  const int64_t row0 = (int64_t)k * T * M + i;
  double sm[KT], sP[KT][KT];                  // walker
  double nm[KT], nP[KT][KT];                  // the others: filtered moments of the next step that they make
  {
    const int64_t e = row0 + (int64_t)max(T - 1 - max(s_own, 0), 0) * M;
    for (int a = 0; a < KT; ++a) {
      sm[a] = nm[a] = io.fmean[e * KT + a];
      for (int b = 0; b < KT; ++b) sP[a][b] = nP[a][b] = io.fcov[(e * KT + a) * KT + b];
    }
  }
  // round it: transitions of tile it, gains of tile it - 1, walk of tile it - 2
  for (int it = 0; it < tiles + 2; ++it) {
    if (s_own >= 0) {
      if (it >= 1 && it <= tiles) {
        const int t = T - 1 - ((it - 1) * kMfTile + s_own);
        double fm[KT], fP[KT][KT], pm[KT], pP[KT][KT], A[K2], Q[K2];
        const double* o = aq + ((it - 1) & 1) * table + ((k - k0) * kMfTile + s_own) * 2 * K2;
        for (int j = 0; j < K2; ++j) { A[j] = o[j]; Q[j] = o[K2 + j]; }
        const int64_t e = row0 + (int64_t)max(t - kMfTile, 0) * M;
        for (int a = 0; a < KT; ++a) {
          fm[a] = nm[a];
          for (int b = 0; b < KT; ++b) fP[a][b] = nP[a][b];
        }
        for (int a = 0; a < KT; ++a) {
          nm[a] = io.fmean[e * KT + a];
          for (int b = 0; b < KT; ++b) nP[a][b] = io.fcov[(e * KT + a) * KT + b];
        }
        mf_predict<KT>(A, Q, fm, fP, pm, pP);
        // G = (A fP)' pP^-1 = fP A' pP^-1
        double AfP[KT][KT], iP[KT][KT], G[KT][KT];
        for (int a = 0; a < KT; ++a)
          for (int b = 0; b < KT; ++b) {
            double w = 0.0;
            for (int q = 0; q < KT; ++q) w = fma(A[a * KT + q], fP[q][b], w);
            AfP[a][b] = w;
          }
        if (KT == 1) {
          iP[0][0] = 1.0 / pP[0][0];
        } else {
          const double det = pP[0][0] * pP[KT - 1][KT - 1] - pP[0][KT - 1] * pP[KT - 1][0];
          iP[0][0] = pP[KT - 1][KT - 1] / det;
          iP[KT - 1][KT - 1] = pP[0][0] / det;
          iP[0][KT - 1] = -pP[0][KT - 1] / det;
          iP[KT - 1][0] = -pP[KT - 1][0] / det;
        }
        for (int a = 0; a < KT; ++a)
          for (int b = 0; b < KT; ++b) {
            double w = 0.0;
            for (int q = 0; q < KT; ++q) w = fma(AfP[q][a], iP[q][b], w);
            G[a][b] = w;
          }
        double* f = fields + (((it - 1) & 1) * kMfTile + s_own) * F * 64 + lane;
        for (int a = 0; a < KT; ++a) {
          f[a * 64] = fm[a];
          f[(KT + a) * 64] = pm[a];
          for (int b = 0; b < KT; ++b) {
            f[(2 * KT + a * KT + b) * 64] = fP[a][b];
            f[(2 * KT + K2 + a * KT + b) * 64] = pP[a][b];
            f[(2 * KT + 2 * K2 + a * KT + b) * 64] = G[a][b];
          }
        }
        if (io.gain && mine && t >= 0)
          for (int j = 0; j < K2; ++j) io.gain[(row0 + (int64_t)t * M) * K2 + j] = G[j / KT][j % KT];
      }
      if (it < tiles)
        mf_transitions<KT>(dm, hy, io.dt, k0, nr, T - 1 - it * kMfTile, -1, aq + (it & 1) * table, threadIdx.x - 64,
                           kMfSmootherT - 64);
    } else if (it >= 2) {
#pragma unroll
      for (int s = 0; s < kMfTile; ++s) {
        const int t = T - 1 - ((it - 2) * kMfTile + s);
        const double* f = fields + ((it & 1) * kMfTile + s) * F * 64 + lane;
        double fm[KT], fP[KT][KT], pm[KT], pP[KT][KT], G[KT][KT];
        for (int a = 0; a < KT; ++a) {
          fm[a] = f[a * 64];
          pm[a] = f[(KT + a) * 64];
          for (int b = 0; b < KT; ++b) {
            fP[a][b] = f[(2 * KT + a * KT + b) * 64];
            pP[a][b] = f[(2 * KT + K2 + a * KT + b) * 64];
            G[a][b] = f[(2 * KT + 2 * K2 + a * KT + b) * 64];
          }
        }
        double dm_[KT], dP[KT][KT], GdP[KT][KT];
        for (int a = 0; a < KT; ++a) {
          dm_[a] = sm[a] - pm[a];
          for (int b = 0; b < KT; ++b) dP[a][b] = sP[a][b] - pP[a][b];
        }
        for (int a = 0; a < KT; ++a) {
          double w = fm[a];
          for (int q = 0; q < KT; ++q) w = fma(G[a][q], dm_[q], w);
          sm[a] = w;
          for (int b = 0; b < KT; ++b) {
            double x = 0.0;
            for (int q = 0; q < KT; ++q) x = fma(G[a][q], dP[q][b], x);
            GdP[a][b] = x;
          }
        }
        for (int a = 0; a < KT; ++a)
          for (int b = 0; b < KT; ++b) {
            double w = fP[a][b];
            for (int q = 0; q < KT; ++q) w = fma(GdP[a][q], G[b][q], w);
            sP[a][b] = w;
          }
        for (int a = 0; a < KT; ++a)
          for (int b = a + 1; b < KT; ++b) sP[a][b] = sP[b][a] = 0.5 * (sP[a][b] + sP[b][a]);
        if (mine && t >= 0) {
          const int64_t kt = (int64_t)k * T + t, e = kt * M + i;
          if (io.hmean) io.hmean[e] = sm[0];
          if (io.hvar) io.hvar[kt * io.var_step + i * io.var_elem] = sP[0][0];
          if (io.smean)
            for (int a = 0; a < KT; ++a) io.smean[e * KT + a] = sm[a];
          if (io.scov)
            for (int j = 0; j < K2; ++j) io.scov[e * K2 + j] = sP[j / KT][j % KT];
        }
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Infinite-horizon space-time filter and smoother (ops.py:796-1068, the filter and
// smoother of InfiniteHorizonGaussianProcess, basemodels.py:1257-1301).  Equispaced steps:
// one A, Q per run (its step size).  Per run:
//   k_ih_tied_part, k_ih_tied
//                 R_tied = (mean_t B' diag(nat2_t) B)^-1 from the whitened form (L L' - 1e-12 I),
//                 partial sums over step ranges on the matrix cores
//   k_ih_dare     `iters` Riccati iterations X <- A (X - X H' S^-1 H X) A' + Q, S = H X H' + R_tied,
//                 from the previous solution; cov = X - K H X (K = X H' S^-1)
//   k_ih_sinv     S_tied, or (heteroscedastic) every step's S_t = H X H' + R_t, inverted; log det
//   k_ih_filter   m_t = A m_{t-1} + X H' S_t^-1 (y_t - H A m_{t-1})
//   k_ih_ell      log N(y_t | H A m_{t-1}, S_t)
//   k_st_gains    (STEADY) G = cov A' X^-1, Qd = cov - G X G'
//   k_st_smoother (ST_STEADY) `iters` iterations X_s <- G X_s G' + Qd from the previous solution
//   k_ih_means    sm_t = fm_t + G (sm_{t+1} - A fm_t) from sm = fm_{T-1}
//   k_ih_spread   H X_s H' at every step
// State layout as in k_st_filter: index c*M + m, H picks the c = 0 block.
// ---------------------------------------------------------------------------
constexpr int kTiedParts = 32;  // step ranges summed in parallel per run

// part[k, p] = sum of L_t L_t' over the p-th of kTiedParts step ranges of run k.
__global__ __launch_bounds__(kT) void k_ih_tied_part(StDims dm, const double* __restrict__ Lw,
                                                     double* __restrict__ part) {
  extern __shared__ double smem[];
  double* pan = smem;                 // 2*kPK*kPS
  double* acc = pan + 2 * kPK * kPS;  // M*M
  const int p = blockIdx.x, k = blockIdx.y, M = dm.M, tid = threadIdx.x;
  const int t0 = (int)((int64_t)dm.T * p / kTiedParts), t1 = (int)((int64_t)dm.T * (p + 1) / kTiedParts);
  for (int e = tid; e < M * M; e += kT) acc[e] = 0.0;
  for (int t = t0; t < t1; ++t) {
    const double* L = Lw + ((int64_t)k * dm.T + t) * M * M;
    wg_gemm_small(M, M, M, 1.0, MatRef{L, M, 1}, MatRef{L, 1, M}, 1.0, acc, M, pan);
  }
  __syncthreads();
  double* out = part + ((int64_t)k * kTiedParts + p) * M * M;
  for (int e = tid; e < M * M; e += kT) out[e] = acc[e];
}

// R_tied = (mean_t L_t L_t' - 1e-12 I)^-1 = (mean_t B' diag(nat2_t) B)^-1, the partial
// sums added in a fixed order.
__global__ __launch_bounds__(kT) void k_ih_tied(StDims dm, const double* __restrict__ part, double* __restrict__ Rt) {
  __shared__ double sL[kMaxM * kMaxM];
  __shared__ double row[2 * kMaxM];
  const int k = blockIdx.x, M = dm.M, tid = threadIdx.x;
  const double it = 1.0 / dm.T;
  for (int e = tid; e < M * M; e += kT) {
    double s = 0.0;
    for (int p = 0; p < kTiedParts; ++p) s += part[((int64_t)k * kTiedParts + p) * M * M + e];
    sL[e] = s * it - ((e / M == e % M) ? kPseudoJitter : 0.0);
  }
  wg_sweep_inv<kMaxM / 16, false>(sL, M, M, row);  // -(tied precision)^-1
  for (int e = tid; e < M * M; e += kT) Rt[(int64_t)k * M * M + e] = -sL[e];
}

struct IhIO {
  const double* aq;    // [K, 2 KT^2] transition of each run's step
  const double* y;     // [K,T,M]
  const double* R;     // [K,T,M,M] (heteroscedastic)
  const double* Rt;    // [K,M,M] tied noise
  double* X;           // [K,D,D] Riccati solution: start in, result out
  double* cov;         // [K,D,D]
  double* STn;         // [K,M,M] -S_tied^-1
  double* ldT;         // [K]
  double* Sn;          // [K,T,M,M] -S_t^-1 (heteroscedastic)
  double* ldS;         // [K,T]
  double* fmean;       // [K,T,D]
  double* ell;         // [K,T]
  int32_t iters, hetero;
};

// Riccati iterations X <- A (X - W W') A' + Q, W = X H' Ls^-T, Ls Ls' = H X H' + R_tied, on the
// filter's register tiles (FilterCore), then cov = X - W W'.  One workgroup per run: the chain of
// iterations bounds it; 12 us an iteration at M = 36, D = 72 (50 us with the sweep inverse and
// products through LDS panels).
template <int KT, int MB>
__global__ __launch_bounds__(128 * MB, 2) void k_ih_dare(StDims dm, IhIO io) {
  using C = FilterCore<KT, MB>;
  constexpr int MP = C::MP, LD = C::LD, NT = C::NT, NR = C::NR, NP = C::NP;
  extern __shared__ double smem[];
  double* X = smem;                    // KT*MP x LD: X H', then W
  double* Lm = X + KT * MP * LD;       // MP x LD
  double* sI = Lm + MP * LD;           // MB of 16 x kDiagLd
  const int M = dm.M, D = dm.D, tid0 = threadIdx.x;
  const int w0 = __builtin_amdgcn_readfirstlane(tid0 >> 6);
  int w = w0, l = tid0 & 63;
  const int k = blockIdx.x;
  const int64_t DD = (int64_t)D * D;
  double A[KT][KT], Q[KT][KT];
#pragma unroll
  for (int a = 0; a < KT; ++a)
#pragma unroll
    for (int b = 0; b < KT; ++b) {
      A[a][b] = io.aq[k * 2 * KT * KT + a * KT + b];
      Q[a][b] = io.aq[k * 2 * KT * KT + KT * KT + a * KT + b];
    }
  typename C::Cov P;
#pragma unroll
  for (int n = 0; n < NP; ++n) {
    int i, j;
    const bool held = C::position(w, n, i, j);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int gi = 16 * i + (l >> 4) + 4 * q, gj = 16 * j + (l & 15);
      const bool on = held && gi < M && gj < M;
#pragma unroll
      for (int a = 0; a < KT; ++a)
#pragma unroll
        for (int b = 0; b < KT; ++b) P[n][a][b][q] = on ? io.X[k * DD + (int64_t)(a * M + gi) * D + b * M + gj] : 0.0;
    }
  }
  tile4 Rt[MB];  // row tile w of the tied noise, identity padding
#pragma unroll
  for (int j = 0; j < MB; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int gi = 16 * w + (l >> 4) + 4 * q, gj = 16 * j + (l & 15);
      Rt[j][q] = w >= MB || j > w ? 0.0 : gi < M && gj < M ? io.Rt[((int64_t)k * M + gi) * M + gj] : gi == gj ? 1.0 : 0.0;
    }
  auto write = [&](double* out) {
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      int i, j;
      if (!C::position(w, n, i, j)) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int gi = 16 * i + (l >> 4) + 4 * q, gj = 16 * j + (l & 15);
        if (gi < M && gj < M) {
#pragma unroll
          for (int a = 0; a < KT; ++a)
#pragma unroll
            for (int b = 0; b < KT; ++b) {
              const int u = a * M + gi, v = b * M + gj;
              out[(int64_t)u * D + v] = P[n][a][b][q];
              if (i != j) out[(int64_t)v * D + u] = P[n][a][b][q];
            }
        }
      }
    }
  };
#pragma unroll 1
  for (int it = 0; it <= io.iters; ++it) {
    w = fresh_s(w0);
    l = fresh_v(tid0) & 63;
    C::publish(P, X, w, l);
    __syncthreads();
    tile4 U[MB], V[MB];
#pragma unroll
    for (int j = 0; j < MB; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        U[j][q] = C::kAllR || w < NR ? X[(16 * w + (l >> 4) + 4 * q) * LD + 16 * j + (l & 15)] : 0.0;
      V[j] = U[j] + Rt[j];
    }
    if (w == 0) {
      tile_store(sI, kDiagLd, 0, 0, V[0], l);
      wave_sync();
      chol16_inverse(sI, kDiagLd, l);
    }
    double quad = 0.0;
    C::template eliminate<false>(P, U, V, quad, X, Lm, sI, nullptr, nullptr, w0, tid0);
    if (it < io.iters) {
      w = fresh_s(w0);
      l = fresh_v(tid0) & 63;
      C::predict(P, A, Q, M, w, l);
      if (it + 1 == io.iters) write(io.X + k * DD);
    } else {
      write(io.cov + k * DD);
    }
    __syncthreads();  // X is read
  }
}

// -S^-1 and log det S, S = H X H' + R: every step's noise, or (TIED) the run's tied noise
template <bool TIED>
__global__ __launch_bounds__(kT) void k_ih_sinv(StDims dm, IhIO io) {
  __shared__ double sS[kMaxM * kMaxM];
  __shared__ double row[2 * kMaxM];
  const int t = blockIdx.x, k = blockIdx.y, M = dm.M, D = dm.D, tid = threadIdx.x;
  const int64_t kt = TIED ? k : (int64_t)k * dm.T + t;
  const double* X = io.X + (int64_t)k * D * D;
  const double* R = (TIED ? io.Rt : io.R) + kt * M * M;
  for (int e = tid; e < M * M; e += kT) sS[e] = R[e] + X[(int64_t)(e / M) * D + e % M];
  const double ld = wg_sweep_inv<kMaxM / 16, true>(sS, M, M, row);
  for (int e = tid; e < M * M; e += kT) (TIED ? io.STn : io.Sn)[kt * M * M + e] = sS[e];
  if (tid == 0) (TIED ? io.ldT : io.ldS)[kt] = ld;
}

constexpr int kAhead = 4;  // steps that the mean recursions load ahead: memory latency is several steps

// m_t = A m_{t-1} + X H' S_t^-1 (y_t - H A m_{t-1}), one workgroup per run: a chain of steps of two
// short products each, bound by their latency.  Eight lanes share an inducing point: they hold
// its row of X H' (all KT components) in registers, S_t^-1's row arrives kAhead steps before it
// is used, and the predicted mean stays with them, so a step is two products, two three-stage
// lane sums and two barriers.  1.2 us a step at M = 36 (4.5 us with one lane a row and S_t^-1 read on
// the way).
template <int KT>
__global__ __launch_bounds__(8 * kMaxM) void k_ih_filter(StDims dm, IhIO io) {
  __shared__ double sv[kMaxM], su[kMaxM];
  const int k = blockIdx.x, M = dm.M, D = dm.D, tid = threadIdx.x, a = tid >> 3, part = tid & 7;
  constexpr int N = kMaxM / 8;
  const double* X = io.X + (int64_t)k * D * D;
  const bool row = a < M;
  double A[KT][KT], xr[KT][N], sr[kAhead][N], yr[kAhead], mp[KT];
#pragma unroll
  for (int c = 0; c < KT; ++c) {
    mp[c] = 0.0;
#pragma unroll
    for (int p = 0; p < KT; ++p) A[c][p] = io.aq[k * 2 * KT * KT + c * KT + p];
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int i = part + 8 * n;
      xr[c][n] = row && i < M ? X[(int64_t)(c * M + a) * D + i] : 0.0;
    }
  }
  const double* y = io.y + (int64_t)k * dm.T * M + (row ? a : 0);
  // S_t^-1's row and y_{t+1}; past the end the last step's again, so that no branch (and no copy
  // that waits for the load) stands between the load and its use
  auto fetch = [&](int t, double (&s)[N], double& yt) {
    t = min(t, dm.T - 1);
    const double* Sn = io.hetero ? io.Sn + ((int64_t)k * dm.T + t) * M * M : io.STn + (int64_t)k * M * M;  // -S^-1
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int j = part + 8 * n;
      s[n] = Sn[row && j < M ? a * M + j : 0];  // used as it comes: sv is 0 from M on
    }
    yt = y[(int64_t)min(t + 1, dm.T - 1) * M];
  };
#pragma unroll
  for (int u = 0; u < kAhead; ++u) fetch(u, sr[u], yr[u]);
  if (part == 0) {
    sv[a] = row ? y[0] : 0.0;
    su[a] = 0.0;
  }
  __syncthreads();
#pragma unroll 1
  for (int t0 = 0; t0 < dm.T; t0 += kAhead) {
#pragma unroll
    for (int b = 0; b < kAhead; ++b) {
      const int t = t0 + b;
      if (t >= dm.T) break;
      double u = 0.0, u1 = 0.0;
#pragma unroll
      for (int n = 0; n < N; n += 2) {
        u = fma(-sr[b][n], sv[part + 8 * n], u);
        u1 = fma(-sr[b][n + 1], sv[part + 8 * n + 8], u1);
      }
      u += u1;
      u += __shfl_xor(u, 1, 64);
      u += __shfl_xor(u, 2, 64);
      u += __shfl_xor(u, 4, 64);
      if (part == 0 && row) su[a] = u;
      const double yt = yr[b];
      fetch(t + kAhead, sr[b], yr[b]);
      __syncthreads();
      double m[KT];
#pragma unroll
      for (int c = 0; c < KT; ++c) {
        double v = 0.0, v1 = 0.0;
#pragma unroll
        for (int n = 0; n < N; n += 2) {
          v = fma(xr[c][n], su[part + 8 * n], v);
          v1 = fma(xr[c][n + 1], su[part + 8 * n + 8], v1);
        }
        v += v1;
        v += __shfl_xor(v, 1, 64);
        v += __shfl_xor(v, 2, 64);
        v += __shfl_xor(v, 4, 64);
        m[c] = mp[c] + v;
      }
      if (part == 0 && row) {
#pragma unroll
        for (int c = 0; c < KT; ++c) io.fmean[((int64_t)k * dm.T + t) * D + c * M + a] = m[c];
      }
#pragma unroll
      for (int c = 0; c < KT; ++c) {
        mp[c] = 0.0;
#pragma unroll
        for (int p = 0; p < KT; ++p) mp[c] = fma(A[c][p], m[p], mp[c]);
      }
      if (part == 0 && row) sv[a] = yt - mp[0];
      __syncthreads();
    }
  }
}

// log N(y_t | H A m_{t-1}, S_t) of every step, one wavefront per (step, run)
template <int KT>
__global__ __launch_bounds__(64) void k_ih_ell(StDims dm, IhIO io) {
  __shared__ double sv[kMaxM];
  const int t = blockIdx.x, k = blockIdx.y, M = dm.M, D = dm.D, l = threadIdx.x;
  const int64_t kt = (int64_t)k * dm.T + t;
  double v = 0.0;
  if (l < M) {
    v = io.y[kt * M + l];
    if (t > 0) {
      for (int p = 0; p < KT; ++p) v = fma(-io.aq[k * 2 * KT * KT + p], io.fmean[(kt - 1) * D + p * M + l], v);
    }
  }
  sv[l] = v;
  __syncthreads();
  const double* Sn = io.hetero ? io.Sn + kt * M * M : io.STn + (int64_t)k * M * M;  // -S^-1
  double u = 0.0;
  if (l < M) {
#pragma unroll 8
    for (int j = 0; j < M; ++j) u = fma(-Sn[j * M + l], sv[j], u);
  }
  double q = u * v;
  for (int o = 32; o > 0; o >>= 1) q += __shfl_xor(q, o, 64);
  if (l == 0) io.ell[kt] = -0.5 * (q + M * kLog2Pi + (io.hetero ? io.ldS[kt] : io.ldT[k]));
}

struct IhSmIO {
  const double* aq;     // [K, 2 KT^2]
  const double* fmean;  // [K,T,D]
  const double* Xs;     // [K,D,D] smoother Riccati solution
  const double* G;      // [K,D,D] gain
  double* pm;           // optional [K,T,M]
  double* pP;           // optional [K,T,M,M]
  double* smean;        // optional [K,T,D]
};

// sm_t = fm_t + G (sm_{t+1} - A fm_t) from sm = fm_{T-1}, one workgroup per run, bound by the latency
// of the chain: four lanes a row with their quarter of G in registers, the filtered means loaded
// kAhead steps before they are used, one barrier a step.  0.7 us a step at D = 72.
template <int KT>
__global__ __launch_bounds__(4 * kMaxD) void k_ih_means(StDims dm, IhSmIO io) {
  __shared__ double sd[2][kMaxD];
  const int k = blockIdx.x, M = dm.M, D = dm.D, T = dm.T, tid = threadIdx.x, r = tid >> 2, part = tid & 3;
  constexpr int N = kMaxD / 4;
  const bool row = r < D;
  const int c = row ? r / M : 0, a = row ? r % M : 0;
  double g[N], Ar[KT];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const int j = part + 4 * n;
    g[n] = row && j < D ? io.G[(int64_t)k * D * D + (int64_t)r * D + j] : 0.0;
  }
#pragma unroll
  for (int p = 0; p < KT; ++p) Ar[p] = io.aq[k * 2 * KT * KT + c * KT + p];
  const double* fm = io.fmean + (int64_t)k * T * D;
  double f[kAhead][KT];  // filtered means of the row's components, kAhead steps
  auto fetch = [&](int t, double (&x)[KT]) {
#pragma unroll
    for (int p = 0; p < KT; ++p) x[p] = fm[(int64_t)(t > 0 ? t : 0) * D + p * M + a];
  };
  auto delta = [&](double ms, const double (&x)[KT]) {  // sm_{t+1} - A fm_t
#pragma unroll
    for (int p = 0; p < KT; ++p) ms = fma(-Ar[p], x[p], ms);
    return row ? ms : 0.0;
  };
#pragma unroll
  for (int u = 0; u < kAhead; ++u) fetch(T - 1 - u, f[u]);
  int cur = 0;
  if (part == 0) {
    double own = f[0][0];
#pragma unroll
    for (int p = 1; p < KT; ++p) own = c == p ? f[0][p] : own;
    sd[0][r] = delta(own, f[0]);
  }
  __syncthreads();
#pragma unroll 1
  for (int s0 = 0; s0 < T; s0 += kAhead) {
#pragma unroll
    for (int b = 0; b < kAhead; ++b) {
      const int t = T - 1 - s0 - b;
      if (t < 0) break;
      double v = 0.0, v1 = 0.0;
#pragma unroll
      for (int n = 0; n < N; n += 2) {
        v = fma(g[n], sd[cur][part + 4 * n], v);
        v1 = fma(g[n + 1], sd[cur][part + 4 * n + 4], v1);
      }
      v += v1;
      v += __shfl_xor(v, 1, 64);
      v += __shfl_xor(v, 2, 64);
      double ms = f[b][0];
#pragma unroll
      for (int p = 1; p < KT; ++p) ms = c == p ? f[b][p] : ms;
      ms += v;
      if (part == 0 && row) {
        const int64_t kt = (int64_t)k * T + t;
        if (io.smean) io.smean[kt * D + r] = ms;
        if (io.pm && r < M) io.pm[kt * M + r] = ms;
      }
      fetch(t - kAhead, f[b]);
      cur ^= 1;
      if (part == 0) sd[cur][r] = delta(ms, f[(b + 1) % kAhead]);
      __syncthreads();
    }
  }
}

// H X_s H' at every step
__global__ __launch_bounds__(kT) void k_ih_spread(StDims dm, IhSmIO io) {
  const int k = blockIdx.y, M = dm.M, D = dm.D;
  const int64_t kt = (int64_t)k * dm.T + blockIdx.x;
  for (int e = threadIdx.x; e < M * M; e += kT)
    io.pP[kt * M * M + e] = io.Xs[(int64_t)k * D * D + (int64_t)(e / M) * D + e % M];
}

// ---------------------------------------------------------------------------
// k_st_predict: MarkovGaussianProcess.predict on the space-time branch
// (basemodels.py:766-816 with temporal_conditional, utils.py:125-141, 185-215), block per
// (test time, run).  The prior is Kronecker in (temporal state) x (latent), so the
// conditional of x(t*) on the two neighbouring smoothed states is P_t (x) I_M, T_t (x) I_M
// with the KT-dim statistics P_t [KT x 2KT], T_t of the temporal kernel (the reference's
// 1e-8 jitter is per diagonal entry either way).  Only H x(t*) is needed:
//   H m* = sum_u P_t[0][u] m_j[u],  S = sum_uv P_t[0][u] P_t[0][v] Sig_j[u][v] + T_t[0][0] I
// over the 2KT M x M blocks of the joint (m_j, Sig_j) of the neighbours (cross block
// G_t P_s,t+1 from the smoother); then f(t*, r) has mean b_r' H m* and variance
// b_r' S b_r + c_r (the diagonal of W P W' + C).  Sentinels at -+1e10 carry (0, Pinf).
// ---------------------------------------------------------------------------
struct StPredIO {
  const double* x;       // [K,T] training times
  const double* xs;      // [K,NS] test times
  const double* B;       // [K,NS,RS,M] spatial conditional rows of the test locations
  const double* cdiag;   // [K,NS,RS]
  const double* smean;   // [K,T,D]
  const double* scov;    // [K,T,D,D]
  const double* scross;  // [K,T,D,D]
  const double* steady;  // [K,D,D] or nullptr: the infinite-horizon state covariance at every test time
  double* mean;          // [K,NS,RS]
  double* var;           // [K,NS,RS]
  int32_t ns, rs;
};

template <int KT>
__global__ __launch_bounds__(kT) void k_st_predict(StDims dm, StHyp hy, StPredIO io) {
  __shared__ double sS[kMaxM * kMaxM];
  __shared__ double hm[kMaxM];
  __shared__ double pc[2 * KT + 1];  // P_t[0][u], then T_t[0][0]
  __shared__ int sidx;
  const int i = blockIdx.x, k = blockIdx.y, M = dm.M, D = dm.D, T = dm.T, tid = threadIdx.x;
  const int64_t DD = (int64_t)D * D;
  const double ls = hy.ls_t[k * hy.stride], var = hy.var_t[k * hy.stride];
  const double* xk = io.x + (int64_t)k * T;
  const double ts = io.xs[(int64_t)k * io.ns + i];
  Model<KT, 0> mdl;
  mdl.init(ls, var, 1.0, 1.0);
  if (tid == 0) {
    // augmented grid [-1e10, x_0 .. x_T-1, 1e10]; ind = searchsorted(left) - 1
    int lo = 0, hi = T;  // first training index with x >= ts
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (xk[mid] < ts) lo = mid + 1;
      else hi = mid;
    }
    const int ind = lo;  // interval (aug[ind], aug[ind + 1]]
    sidx = ind;
    const double xl = ind == 0 ? -1e10 : xk[ind - 1];
    const double xr = ind == T ? 1e10 : xk[ind];
    double Af[KT][KT], Qf[KT][KT], Ab[KT][KT], Qb[KT][KT];
    mdl.discretise(ts - xl, Af, Qf);
    mdl.discretise(xr - ts, Ab, Qb);
    // Q-+ = Qb + Ab Qf Ab' + 1e-8 I ; V = Q-+^-1 Ab ; T = Qf - (Ab Qf)' V Qf ; W = Qf V'
    double AQ[KT][KT], Qm[KT][KT], V[KT][KT], W[KT][KT], Pt[KT][2 * KT];
    for (int a = 0; a < KT; ++a)
      for (int b = 0; b < KT; ++b) {
        double s = 0.0;
        for (int q = 0; q < KT; ++q) s = fma(Ab[a][q], Qf[q][b], s);
        AQ[a][b] = s;
      }
    for (int a = 0; a < KT; ++a)
      for (int b = 0; b < KT; ++b) {
        double s = Qb[a][b] + (a == b ? 1e-8 : 0.0);
        for (int q = 0; q < KT; ++q) s = fma(AQ[a][q], Ab[b][q], s);
        Qm[a][b] = s;
      }
    double iQ[KT][KT];
    if (KT == 1) {
      iQ[0][0] = 1.0 / Qm[0][0];
    } else {
      const double det = Qm[0][0] * Qm[KT - 1][KT - 1] - Qm[0][KT - 1] * Qm[KT - 1][0];
      iQ[0][0] = Qm[KT - 1][KT - 1] / det;
      iQ[KT - 1][KT - 1] = Qm[0][0] / det;
      iQ[0][KT - 1] = -Qm[0][KT - 1] / det;
      iQ[KT - 1][0] = -Qm[KT - 1][0] / det;
    }
    for (int a = 0; a < KT; ++a)
      for (int b = 0; b < KT; ++b) {
        double s = 0.0;
        for (int q = 0; q < KT; ++q) s = fma(iQ[a][q], Ab[q][b], s);
        V[a][b] = s;
      }
    for (int a = 0; a < KT; ++a)
      for (int b = 0; b < KT; ++b) {
        double s = 0.0;
        for (int q = 0; q < KT; ++q) s = fma(Qf[a][q], V[b][q], s);
        W[a][b] = s;
      }
    double WAb[KT][KT];
    for (int a = 0; a < KT; ++a)
      for (int b = 0; b < KT; ++b) {
        double s = 0.0;
        for (int q = 0; q < KT; ++q) s = fma(W[a][q], Ab[q][b], s);
        WAb[a][b] = s;
      }
    for (int a = 0; a < KT; ++a)
      for (int b = 0; b < KT; ++b) {
        double s = Af[a][b];
        for (int q = 0; q < KT; ++q) s = fma(-WAb[a][q], Af[q][b], s);
        Pt[a][b] = s;
        Pt[a][KT + b] = W[a][b];
      }
    // T[0][0] = Qf[0][0] - (Ab Qf)[:,0]' V Qf[:,0]
    double VQ[KT];
    for (int a = 0; a < KT; ++a) {
      double s = 0.0;
      for (int q = 0; q < KT; ++q) s = fma(V[a][q], Qf[q][0], s);
      VQ[a] = s;
    }
    double t00 = Qf[0][0];
    for (int a = 0; a < KT; ++a) t00 = fma(-AQ[a][0], VQ[a], t00);
    for (int u = 0; u < 2 * KT; ++u) pc[u] = Pt[0][u];
    pc[2 * KT] = t00;
  }
  __syncthreads();
  const int ind = sidx;
  const bool lsent = ind == 0, rsent = ind == T;
  const int64_t tl = (int64_t)k * T + (lsent ? 0 : ind - 1), tr = (int64_t)k * T + (rsent ? T - 1 : ind);
  const double* mL = io.smean + tl * D;
  const double* mR = io.smean + tr * D;
  const double* PL = io.steady ? nullptr : io.scov + tl * DD;
  const double* PR = io.steady ? nullptr : io.scov + tr * DD;
  const double* Cx = io.steady ? nullptr : io.scross + tl * DD;  // Cov(left, right); 0 after the left sentinel
  for (int a = tid; a < M; a += kT) {
    double s = 0.0;
    for (int c = 0; c < KT; ++c) {
      if (!lsent) s = fma(pc[c], mL[c * M + a], s);
      if (!rsent) s = fma(pc[KT + c], mR[c * M + a], s);
    }
    hm[a] = s;
  }
  if (io.steady) {
    // temporal_conditional_infinite_horizon (utils.py:163-177): the smoother's steady
    // covariance replaces the conditional one
    for (int e = tid; e < M * M; e += kT) sS[e] = io.steady[k * DD + (int64_t)(e / M) * D + e % M];
  } else
  for (int e = tid; e < M * M; e += kT) {
    const int a = e / M, b = e % M;
    double s = (a == b) ? pc[2 * KT] : 0.0;
    for (int c = 0; c < KT; ++c)
      for (int c2 = 0; c2 < KT; ++c2) {
        const int64_t ia = (int64_t)(c * M + a) * D, ib = (int64_t)(c2 * M + b) * D;
        const double wl = pc[c], wr = pc[KT + c], vl = pc[c2], vr = pc[KT + c2];
        const double pl = lsent ? (a == b ? mdl.Pinf[c][c2] : 0.0) : PL[ia + c2 * M + b];
        const double pr = rsent ? (a == b ? mdl.Pinf[c][c2] : 0.0) : PR[ia + c2 * M + b];
        const double xlr = lsent ? 0.0 : Cx[ia + c2 * M + b];   // Cov(left_a, right_b)
        const double xrl = lsent ? 0.0 : Cx[ib + c * M + a];    // Cov(right_a, left_b)
        s = fma(wl * vl, pl, s);
        s = fma(wr * vr, pr, s);
        s = fma(wl * vr, xlr, s);
        s = fma(wr * vl, xrl, s);
      }
    sS[e] = s;
  }
  __syncthreads();
  const int64_t base = ((int64_t)k * io.ns + i) * io.rs;
  for (int r = tid; r < io.rs; r += kT) {
    const double* b = io.B + (base + r) * M;
    double mu = 0.0, v = io.cdiag[base + r];
    for (int a = 0; a < M; ++a) {
      const double ba = b[a];
      mu = fma(ba, hm[a], mu);
      double u = 0.0;
      for (int c = 0; c < M; ++c) u = fma(sS[a * M + c], b[c], u);
      v = fma(ba, u, v);
    }
    io.mean[base + r] = mu;
    io.var[base + r] = v;
  }
}

constexpr size_t kPseudoSmem = sizeof(double) * (2 * kPK * kPS + kMaxM * kMaxM + 3 * kMaxM);
constexpr size_t kTiedSmem = sizeof(double) * (2 * kPK * kPS + kMaxM * kMaxM);
constexpr size_t kSitesSmem =
    sizeof(double) * (2 * kMaxM * kSLd + 5 * kMaxM + 4 * 32 + 4);
static_assert(2 * kSitesSmem <= 160 * 1024, "two workgroups of k_st_sites a CU");
constexpr size_t kOrderedSmem =
    sizeof(double) * (2 * kPK * kPS + 2 * kRC * kLC + 2 * kMaxM + kRC + 2 * kMaxM + 4);
constexpr size_t kCavitySmem = sizeof(double) * (2 * kPK * kPS + 2 * kMaxM * kMaxM + 4 * kMaxM + 4);

int check_dims(const bn_st_dims* d, StDims& dm) {
  if (d == nullptr) return st_fail(BN_EINVAL, "dims is NULL");
  if (d->n_runs < 1 || d->n_steps < 1 || d->n_loc < 1) return st_fail(BN_EINVAL, "empty space-time problem");
  if (d->n_inducing < 1 || d->n_inducing > kMaxM)
    return st_fail(BN_EUNSUPPORTED, "number of spatial inducing points must be in [1, 64]");
  if (d->temporal_kind != BN_MATERN12 && d->temporal_kind != BN_MATERN32)
    return st_fail(BN_EUNSUPPORTED, "space-time temporal kernel must be Matern12 or Matern32");
  dm.K = d->n_runs;
  dm.T = d->n_steps;
  dm.R = d->n_loc;
  dm.M = d->n_inducing;
  dm.KT = d->temporal_kind;  // state dimension of the temporal component
  dm.D = dm.KT * dm.M;
  return BN_OK;
}

StHyp make_hyp(const bn_st_hypers* h) { return StHyp{h->ls_t, h->var_t, h->var_s, h->stride}; }

template <int KT, int MB>
int smoother_attr() {
  const int n = (int)sizeof(double) * StTiles<KT, MB>::SMEM;
  ST_HIP_CHECK(hipFuncSetAttribute((const void*)k_ih_dare<KT, MB>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)sizeof(double) * filter_smem(KT, MB)));
  for (const void* f : {(const void*)k_st_gains<KT, MB, false>, (const void*)k_st_gains<KT, MB, true>,
                        (const void*)k_st_chain<KT, MB>, (const void*)k_st_smoother<KT, MB, ST_STEADY>,
                        (const void*)k_st_smoother<KT, MB, ST_WALK>, (const void*)k_st_smoother<KT, MB, ST_COMPOSE>,
                        (const void*)k_st_smoother<KT, MB, ST_JOIN>})
    ST_HIP_CHECK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, n));
  return BN_OK;
}

// Dynamic LDS above the default limit is opted into once per kernel.
int set_smem_limits() {
  static int done = 0;
  if (done) return BN_OK;
#define ST_FILTER_ATTR(KT, MB)                                                                                  \
  ST_HIP_CHECK(hipFuncSetAttribute((const void*)k_st_filter<KT, MB>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                   (int)sizeof(double) * filter_smem(KT, MB)));                                        \
  if (int rc = smoother_attr<KT, MB>()) return rc
  ST_FILTER_ATTR(1, 1);
  ST_FILTER_ATTR(1, 2);
  ST_FILTER_ATTR(1, 3);
  ST_FILTER_ATTR(1, 4);
  ST_FILTER_ATTR(2, 1);
  ST_FILTER_ATTR(2, 2);
  ST_FILTER_ATTR(2, 3);
  ST_FILTER_ATTR(2, 4);
#undef ST_FILTER_ATTR
#define ST_SITES_ATTR1(KERNEL, MT, MD, KD, N)                                                                       \
  ST_HIP_CHECK(hipFuncSetAttribute((const void*)KERNEL<MT, MD, KD>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)N))
#define ST_SITES_ATTR(KERNEL, MT, MD, N)                    \
  ST_SITES_ATTR1(KERNEL, MT, MD, LIK_GAUSSIAN, N);          \
  ST_SITES_ATTR1(KERNEL, MT, MD, LIK_BERNOULLI_PROBIT, N);  \
  ST_SITES_ATTR1(KERNEL, MT, MD, LIK_POISSON, N);           \
  ST_SITES_ATTR1(KERNEL, MT, MD, LIK_STUDENTS_T, N)
  ST_HIP_CHECK(hipFuncSetAttribute((const void*)k_mf_smoother<1>, hipFuncAttributeMaxDynamicSharedMemorySize, 163840));
  ST_HIP_CHECK(hipFuncSetAttribute((const void*)k_mf_smoother<2>, hipFuncAttributeMaxDynamicSharedMemorySize, 163840));
  ST_HIP_CHECK(hipFuncSetAttribute((const void*)k_mf_pseudo, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)kPseudoSmem));
  ST_SITES_ATTR(k_st_sites, M_VI, BN_ST_UPDATE, kSitesSmem);
  ST_SITES_ATTR(k_st_sites, M_VI, BN_ST_ENERGY, kSitesSmem);
  ST_SITES_ATTR1(k_st_sites, M_VI, BN_ST_PROJECT, 0, kSitesSmem);
  ST_SITES_ATTR(k_st_sites, M_NEWTON, BN_ST_UPDATE, kSitesSmem);
  ST_SITES_ATTR(k_st_sites, M_NEWTON, BN_ST_ENERGY, kSitesSmem);
  ST_SITES_ATTR(k_st_sites, M_EP, BN_ST_ENERGY, kSitesSmem);
  ST_SITES_ATTR(k_st_sites_ordered, M_VI, BN_ST_UPDATE, kOrderedSmem);
  ST_SITES_ATTR1(k_st_sites_ordered, M_VI, BN_ST_PROJECT, 0, kOrderedSmem);
  ST_SITES_ATTR(k_st_sites_ordered, M_NEWTON, BN_ST_UPDATE, kOrderedSmem);
  ST_SITES_ATTR(k_st_sites_ordered, M_EP, BN_ST_UPDATE, kOrderedSmem);
#undef ST_SITES_ATTR
#undef ST_SITES_ATTR1
  ST_HIP_CHECK(hipFuncSetAttribute((const void*)k_st_ep_cavity<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)kCavitySmem));
  ST_HIP_CHECK(hipFuncSetAttribute((const void*)k_st_ep_cavity<true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)kCavitySmem));
  done = 1;
  return BN_OK;
}

// k_st_filter for the 16-wide tiles that M needs.
template <int KT>
void launch_st_filter(hipStream_t st, StDims dm, StHyp hy, StFilterIO io) {
  switch ((dm.M + 15) / 16) {
    case 1:
      hipLaunchKernelGGL((k_st_filter<KT, 1>), dim3(dm.K), dim3(128), sizeof(double) * filter_smem(KT, 1), st, dm, hy, io);
      break;
    case 2:
      hipLaunchKernelGGL((k_st_filter<KT, 2>), dim3(dm.K), dim3(256), sizeof(double) * filter_smem(KT, 2), st, dm, hy, io);
      break;
    case 3:
      hipLaunchKernelGGL((k_st_filter<KT, 3>), dim3(dm.K), dim3(384), sizeof(double) * filter_smem(KT, 3), st, dm, hy, io);
      break;
    default:
      hipLaunchKernelGGL((k_st_filter<KT, 4>), dim3(dm.K), dim3(512), sizeof(double) * filter_smem(KT, 4), st, dm, hy, io);
      break;
  }
}

template <int KT>
void launch_st_transitions(hipStream_t st, StDims dm, StHyp hy, const double* dt, double* aq) {
  const unsigned nb = (unsigned)(((int64_t)dm.K * dm.T + kT - 1) / kT);
  hipLaunchKernelGGL(k_st_transitions<KT>, dim3(nb), dim3(kT), 0, st, dm, hy, dt, aq);
}

// The backward pass over blocks of steps from the end of the runs.
template <int KT, int MB>
int launch_st_smoother(hipStream_t st, StDims dm, StHyp hy, const double* aq, const double* fmean, const double* fcov,
                       StSmootherIO io) {
  using S = StTiles<KT, MB>;
  const unsigned nt = 64 * S::NR;
  const size_t smem = sizeof(double) * S::SMEM;
  hipLaunchKernelGGL((k_st_terminal<KT, MB>), dim3(dm.K), dim3(kT), 0, st, dm, hy, fmean, fcov, io);
  for (int t1 = dm.T - 1; t1 > 0; t1 = io.t0) {  // steps [t0, t1)
    io.t0 = t1 > io.tb ? t1 - io.tb : 0;
    io.nb = t1 - io.t0;
    io.nc = smoother_chunks(dm, io.nb);
    const StGainIO gi{aq, fmean, fcov, io.rec, io.t0, io.tb, nullptr, nullptr};
    hipLaunchKernelGGL((k_st_gains<KT, MB, false>), dim3(io.nb, dm.K), dim3(nt), smem, st, dm, gi);
    if (io.nc > 1) {
      hipLaunchKernelGGL((k_st_chain<KT, MB>), dim3(io.nc - 1, dm.K), dim3(nt), smem, st, io);
      hipLaunchKernelGGL((k_st_smoother<KT, MB, ST_COMPOSE>), dim3(io.nc - 1, dm.K), dim3(nt), smem, st, dm, io);
      hipLaunchKernelGGL((k_st_smoother<KT, MB, ST_JOIN>), dim3(1, dm.K), dim3(nt), smem, st, dm, io);
    }
    hipLaunchKernelGGL((k_st_smoother<KT, MB, ST_WALK>), dim3(io.nc, dm.K), dim3(nt), smem, st, dm, io);
    ST_HIP_CHECK(hipGetLastError());
    io.in = 1 - io.in;
  }
  return BN_OK;
}

template <int KT>
int launch_st_smoother(hipStream_t st, StDims dm, StHyp hy, const double* dt, double* aq, const double* fmean,
                       const double* fcov, StSmootherIO io) {
  launch_st_transitions<KT>(st, dm, hy, dt, aq);
  switch ((dm.M + 15) / 16) {
    case 1: return launch_st_smoother<KT, 1>(st, dm, hy, aq, fmean, fcov, io);
    case 2: return launch_st_smoother<KT, 2>(st, dm, hy, aq, fmean, fcov, io);
    case 3: return launch_st_smoother<KT, 3>(st, dm, hy, aq, fmean, fcov, io);
    default: return launch_st_smoother<KT, 4>(st, dm, hy, aq, fmean, fcov, io);
  }
}

// Doubles at the head of the infinite-horizon workspace: transitions, the smoother's map and gain.
int64_t ih_head(const StDims& dm) {
  return (int64_t)dm.K * (2 * dm.KT * dm.KT + map_doubles(dm) + (int64_t)dm.D * dm.D);
}

// The transition of each run's step: one step a run.
void launch_ih_transitions(hipStream_t st, StDims dm, StHyp hy, const double* step, double* aq) {
  dm.T = 1;
  if (dm.KT == 1) launch_st_transitions<1>(st, dm, hy, step, aq);
  else launch_st_transitions<2>(st, dm, hy, step, aq);
}

template <int KT, int MB>
void launch_ih_dare(hipStream_t st, StDims dm, IhIO io) {
  hipLaunchKernelGGL((k_ih_dare<KT, MB>), dim3(dm.K), dim3(128 * MB), sizeof(double) * filter_smem(KT, MB), st, dm, io);
}
template <int KT>
void launch_ih_dare(hipStream_t st, StDims dm, IhIO io) {
  switch ((dm.M + 15) / 16) {
    case 1: return launch_ih_dare<KT, 1>(st, dm, io);
    case 2: return launch_ih_dare<KT, 2>(st, dm, io);
    case 3: return launch_ih_dare<KT, 3>(st, dm, io);
    default: return launch_ih_dare<KT, 4>(st, dm, io);
  }
}

template <int KT, int MB>
void launch_ih_smoother(hipStream_t st, StDims dm, StGainIO gi, StSmootherIO si) {
  using S = StTiles<KT, MB>;
  const size_t smem = sizeof(double) * S::SMEM;
  hipLaunchKernelGGL((k_st_gains<KT, MB, true>), dim3(1, dm.K), dim3(64 * S::NR), smem, st, dm, gi);
  if (si.iters > 0)
    hipLaunchKernelGGL((k_st_smoother<KT, MB, ST_STEADY>), dim3(1, dm.K), dim3(64 * S::NR), smem, st, dm, si);
}
template <int KT>
void launch_ih_smoother(hipStream_t st, StDims dm, StGainIO gi, StSmootherIO si) {
  switch ((dm.M + 15) / 16) {
    case 1: return launch_ih_smoother<KT, 1>(st, dm, gi, si);
    case 2: return launch_ih_smoother<KT, 2>(st, dm, gi, si);
    case 3: return launch_ih_smoother<KT, 3>(st, dm, gi, si);
    default: return launch_ih_smoother<KT, 4>(st, dm, gi, si);
  }
}

// k_st_sites / k_st_sites_ordered for the likelihood kind L.kind (checked by check_lik).
#define ST_SITES_LAUNCH(KERNEL, KD, N)                                                                              \
  hipLaunchKernelGGL((KERNEL<MT, MD, KD>), grid, dim3(kT), N, st, dm, L, gh, io, lr, ensure_psd, power, mask_pseudo)
#define ST_SITES_SWITCH(KERNEL, N)                                                        \
  switch (L.kind) {                                                                       \
    case LIK_GAUSSIAN: ST_SITES_LAUNCH(KERNEL, LIK_GAUSSIAN, N); break;                   \
    case LIK_BERNOULLI_PROBIT: ST_SITES_LAUNCH(KERNEL, LIK_BERNOULLI_PROBIT, N); break;   \
    case LIK_POISSON: ST_SITES_LAUNCH(KERNEL, LIK_POISSON, N); break;                     \
    default: ST_SITES_LAUNCH(KERNEL, LIK_STUDENTS_T, N); break;                           \
  }
template <int MT, int MD>
void launch_st_sites(dim3 grid, hipStream_t st, StDims dm, LikParams L, GHTable gh, StSiteIO io, double lr,
                     int ensure_psd, double power, int mask_pseudo) {
  ST_SITES_SWITCH(k_st_sites, kSitesSmem)
}
template <int MT>
void launch_st_update_ordered(dim3 grid, hipStream_t st, StDims dm, LikParams L, GHTable gh, StSiteIO io, double lr,
                              int ensure_psd, double power, int mask_pseudo) {
  constexpr int MD = BN_ST_UPDATE;
  ST_SITES_SWITCH(k_st_sites_ordered, kOrderedSmem)
}
#undef ST_SITES_SWITCH
#undef ST_SITES_LAUNCH

// bn_st_sites (whitened = false) and bn_st_sites_whitened.
int st_sites(bool whitened, const bn_st_dims* dims, const bn_lik_desc* lik, int32_t method, int32_t mode,
             int32_t gh_points, double lr, int32_t ensure_psd, const float* y, const double* B, const double* cdiag,
             const double* post_mean, const double* post_cov, const float* batch, double* nat1, double* nat2,
             double* Lw, double* zw, double* ldl, double* part0, double* part1, float* out_mean, float* out_jac,
             float* out_hess, void* stream) {
  StDims dm;
  if (int rc = check_dims(dims, dm)) return rc;
  if (!lik || !y || !B || !cdiag || !post_mean || !post_cov || !nat1 || !nat2 || !Lw || !zw || !ldl || !part0 ||
      !part1)
    return st_fail(BN_EINVAL, "NULL argument to bn_st_sites");
  if (method != BN_VI && method != BN_NEWTON)
    return st_fail(BN_EUNSUPPORTED, "space-time sites support BN_VI and BN_NEWTON");
  if (mode != BN_ST_UPDATE && mode != BN_ST_ENERGY && mode != BN_ST_PROJECT)
    return st_fail(BN_EINVAL, "mode must be BN_ST_UPDATE, BN_ST_ENERGY or BN_ST_PROJECT");
  LikParams L;
  if (int rc = check_lik(lik, L)) return rc;
  GHTable gh;
  if (int rc = make_gh_table(gh_points, gh)) return rc;
  if (int rc = set_smem_limits()) return rc;
  StSiteIO io{y,    B,    cdiag, post_mean, post_cov, nat1,    nat2,     Lw,
              zw,   ldl,  part0, part1,     out_mean, out_jac, out_hess, batch};
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid(dm.T, dm.K);
  BN_TIMED(KID_ST_SITES, st);
  if (mode == BN_ST_PROJECT) {
    // the projection is method- and likelihood-free
    if (whitened)
      hipLaunchKernelGGL((k_st_sites<M_VI, BN_ST_PROJECT, 0>), grid, dim3(kT), kSitesSmem, st, dm, L, gh, io, lr,
                         ensure_psd, 1.0, 0);
    else
      hipLaunchKernelGGL((k_st_sites_ordered<M_VI, BN_ST_PROJECT, 0>), grid, dim3(kT), kOrderedSmem, st, dm, L, gh, io,
                         lr, ensure_psd, 1.0, 0);
  } else if (mode == BN_ST_ENERGY) {
    if (method == BN_VI) launch_st_sites<M_VI, BN_ST_ENERGY>(grid, st, dm, L, gh, io, lr, ensure_psd, 1.0, 0);
    else launch_st_sites<M_NEWTON, BN_ST_ENERGY>(grid, st, dm, L, gh, io, lr, ensure_psd, 1.0, 0);
  } else if (whitened) {
    if (method == BN_VI) launch_st_sites<M_VI, BN_ST_UPDATE>(grid, st, dm, L, gh, io, lr, ensure_psd, 1.0, 0);
    else launch_st_sites<M_NEWTON, BN_ST_UPDATE>(grid, st, dm, L, gh, io, lr, ensure_psd, 1.0, 0);
  } else {
    if (method == BN_VI) launch_st_update_ordered<M_VI>(grid, st, dm, L, gh, io, lr, ensure_psd, 1.0, 0);
    else launch_st_update_ordered<M_NEWTON>(grid, st, dm, L, gh, io, lr, ensure_psd, 1.0, 0);
  }
  ST_HIP_CHECK(hipGetLastError());
  return BN_OK;
}

}  // namespace

extern "C" {

int bn_st_conditional(const bn_st_dims* dims, const bn_st_hypers* hyp, int32_t spatial_kind, double ls_s, const double* z,
                      const double* Lzz, const float* r, double* B, double* cdiag, void* stream) {
  StDims dm;
  if (int rc = check_dims(dims, dm)) return rc;
  if (!hyp || !z || !Lzz || !r || !B || !cdiag) return st_fail(BN_EINVAL, "NULL argument to bn_st_conditional");
  if (!(ls_s > 0)) return st_fail(BN_EINVAL, "spatial lengthscale must be > 0");
  if (spatial_kind < BN_MATERN12 || spatial_kind > BN_MATERN52)
    return st_fail(BN_EUNSUPPORTED, "spatial kernel must be Matern12, Matern32 or Matern52");
  hipStream_t st = (hipStream_t)stream;
  BN_TIMED(KID_ST_CONDITIONAL, st);
  hipLaunchKernelGGL(k_st_conditional, dim3(dm.T, dm.K), dim3(kT), 0, st, dm, make_hyp(hyp), Lzz, z, spatial_kind, ls_s, r, B,
                     cdiag);
  ST_HIP_CHECK(hipGetLastError());
  return BN_OK;
}

int bn_st_sites(const bn_st_dims* dims, const bn_lik_desc* lik, int32_t method, int32_t mode, int32_t gh_points,
                double lr, int32_t ensure_psd, const float* y, const double* B, const double* cdiag,
                const double* post_mean, const double* post_cov, const float* batch, double* nat1, double* nat2,
                double* Lw, double* zw, double* ldl, double* part0, double* part1, float* out_mean, float* out_jac,
                float* out_hess, void* stream) {
  return st_sites(false, dims, lik, method, mode, gh_points, lr, ensure_psd, y, B, cdiag, post_mean, post_cov, batch, nat1,
                  nat2, Lw, zw, ldl, part0, part1, out_mean, out_jac, out_hess, stream);
}

int bn_st_sites_whitened(const bn_st_dims* dims, const bn_lik_desc* lik, int32_t method, int32_t mode, int32_t gh_points,
                double lr, int32_t ensure_psd, const float* y, const double* B, const double* cdiag,
                const double* post_mean, const double* post_cov, const float* batch, double* nat1, double* nat2,
                double* Lw, double* zw, double* ldl, double* part0, double* part1, float* out_mean, float* out_jac,
                float* out_hess, void* stream) {
  return st_sites(true, dims, lik, method, mode, gh_points, lr, ensure_psd, y, B, cdiag, post_mean, post_cov, batch, nat1,
                  nat2, Lw, zw, ldl, part0, part1, out_mean, out_jac, out_hess, stream);
}

int bn_st_ep_sites(const bn_st_dims* dims, const bn_lik_desc* lik, int32_t mode, int32_t gh_points, double lr,
                   int32_t ensure_psd, double power, const float* y, const double* B, const double* cdiag,
                   const double* post_mean, const double* post_cov, double* nat1, double* nat2, double* Lw,
                   double* zw, double* ldl, double* cav_mean, double* cav_cov, double* part0, double* part1,
                   float* out_mean, float* out_jac, float* out_hess, void* stream) {
  StDims dm;
  if (int rc = check_dims(dims, dm)) return rc;
  if (!lik || !y || !B || !cdiag || !post_mean || !post_cov || !nat1 || !nat2 || !Lw || !zw || !ldl || !cav_mean ||
      !cav_cov || !part0 || !part1)
    return st_fail(BN_EINVAL, "NULL argument to bn_st_ep_sites");
  if (mode != BN_ST_UPDATE && mode != BN_ST_ENERGY)
    return st_fail(BN_EINVAL, "mode must be BN_ST_UPDATE or BN_ST_ENERGY (the projection is method-free: bn_st_sites)");
  if (!(power > 0.0 && power <= 1.0)) return st_fail(BN_EINVAL, "EP power must be in (0, 1]");
  LikParams L;
  if (int rc = check_lik(lik, L)) return rc;
  if (dm.R > 1 && L.kind != LIK_GAUSSIAN)
    return st_fail(BN_EUNSUPPORTED,
                   "EP with several locations per step moment-matches all of them jointly; only the Gaussian "
                   "likelihood has that in closed form (one location per step takes any likelihood)");
  if (dm.R > 1 && mode == BN_ST_ENERGY)
    return st_fail(BN_EUNSUPPORTED, "masking in spatio-temporal models not implemented for EP");
  GHTable gh;
  if (int rc = make_gh_table(gh_points, gh)) return rc;
  if (int rc = set_smem_limits()) return rc;
  // basemodels.py:138-144, 653: the pseudo observations are masked only when their
  // dimension (M) equals the data's (R)
  const int mask_pseudo = dm.M == dm.R ? 1 : 0;
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid(dm.T, dm.K);
  StCavityIO cio{y, post_mean, post_cov, Lw, zw, ldl, cav_mean, cav_cov, part1};
  StSiteIO io{y,  B,   cdiag, cav_mean, cav_cov,  nat1,    nat2,     Lw,
              zw, ldl, part0, part1,    out_mean, out_jac, out_hess, nullptr};
  BN_TIMED(KID_ST_SITES, st);
  if (mode == BN_ST_UPDATE) {
    hipLaunchKernelGGL((k_st_ep_cavity<false>), grid, dim3(kT), kCavitySmem, st, dm, cio, power, mask_pseudo);
    launch_st_update_ordered<M_EP>(grid, st, dm, L, gh, io, lr, ensure_psd, power, mask_pseudo);
  } else {
    hipLaunchKernelGGL((k_st_ep_cavity<true>), grid, dim3(kT), kCavitySmem, st, dm, cio, power, mask_pseudo);
    launch_st_sites<M_EP, BN_ST_ENERGY>(grid, st, dm, L, gh, io, lr, ensure_psd, power, mask_pseudo);
  }
  ST_HIP_CHECK(hipGetLastError());
  return BN_OK;
}

int64_t bn_st_workspace_bytes(const bn_st_dims* dims) {
  StDims dm;
  if (check_dims(dims, dm) != BN_OK) return -1;
  // per run: the transitions of every step (2 KT^2); then, for the filter, the determinant of every
  // step (2) or, for the smoother, its states, chunk maps and block of maps
  const int64_t nc = smoother_max_chunks(dm);
  const int64_t smoother = (2 + nc) * state_doubles(dm) + (nc + gain_block_steps(dm)) * map_doubles(dm);
  const int64_t filter = 2 * (int64_t)dm.T;
  return (int64_t)dm.K * (2 * (int64_t)dm.KT * dm.KT * dm.T + (smoother > filter ? smoother : filter)) *
             (int64_t)sizeof(double) + 4096;
}

int bn_st_filter(const bn_st_dims* dims, const bn_st_hypers* hyp, const double* dt, const double* Lw,
                 const double* zw, const double* ldl, double* filter_mean, double* filter_cov, double* ell_steps,
                 double* loglik, void* workspace, void* stream) {
  StDims dm;
  if (int rc = check_dims(dims, dm)) return rc;
  if (!hyp || !dt || !Lw || !zw || !ldl || !filter_mean || !filter_cov || !ell_steps || !loglik || !workspace)
    return st_fail(BN_EINVAL, "NULL argument to bn_st_filter");
  double* ws = (double*)workspace;
  if (int rc = set_smem_limits()) return rc;
  StFilterIO io{ws, Lw, zw, filter_mean, filter_cov, ell_steps, ws + (int64_t)dm.K * dm.T * 2 * dm.KT * dm.KT};
  hipStream_t st = (hipStream_t)stream;
  const StHyp hy = make_hyp(hyp);
  {
    BN_TIMED(KID_ST_FILTER, st);
    if (dm.KT == 1) {
      launch_st_transitions<1>(st, dm, hy, dt, ws);
      launch_st_filter<1>(st, dm, hy, io);
    } else {
      launch_st_transitions<2>(st, dm, hy, dt, ws);
      launch_st_filter<2>(st, dm, hy, io);
    }
    hipLaunchKernelGGL(k_st_ell, dim3((unsigned)(((int64_t)dm.K * dm.T + kT - 1) / kT)), dim3(kT), 0, st, dm, io.det,
                       ldl, ell_steps);
  }
  ST_HIP_CHECK(hipGetLastError());
  {
    BN_TIMED(KID_ST_SUM, st);
    hipLaunchKernelGGL(k_st_sum, dim3(dm.K), dim3(kT), 0, st, dm.T, ell_steps, loglik);
  }
  ST_HIP_CHECK(hipGetLastError());
  return BN_OK;
}

int bn_st_smoother(const bn_st_dims* dims, const bn_st_hypers* hyp, const double* dt, const double* filter_mean,
                   const double* filter_cov, double* post_mean, double* post_cov, void* workspace, void* stream) {
  return bn_st_smoother_full(dims, hyp, dt, filter_mean, filter_cov, post_mean, post_cov, nullptr, nullptr, nullptr,
                             workspace, stream);
}

int bn_st_smoother_full(const bn_st_dims* dims, const bn_st_hypers* hyp, const double* dt, const double* filter_mean,
                        const double* filter_cov, double* post_mean, double* post_cov, double* smooth_mean,
                        double* smooth_cov, double* smooth_cross, void* workspace, void* stream) {
  StDims dm;
  if (int rc = check_dims(dims, dm)) return rc;
  if (!hyp || !dt || !filter_mean || !filter_cov || !post_mean || !post_cov || !workspace)
    return st_fail(BN_EINVAL, "NULL argument to bn_st_smoother");
  if ((smooth_mean == nullptr) != (smooth_cov == nullptr) || (smooth_mean == nullptr) != (smooth_cross == nullptr))
    return st_fail(BN_EINVAL, "bn_st_smoother_full: smooth_mean, smooth_cov and smooth_cross go together");
  if (int rc = set_smem_limits()) return rc;
  const int64_t K = dm.K;
  const int nc = smoother_max_chunks(dm);
  // transitions, states, chunk maps, the block's maps (bn_st_workspace_bytes)
  double* aq = (double*)workspace;
  StSmootherIO io{};
  io.state = aq + K * dm.T * 2 * dm.KT * dm.KT;
  io.slots = 2 + nc;
  io.comp = io.state + K * io.slots * state_doubles(dm);
  io.rec = io.comp + K * nc * map_doubles(dm);
  io.tb = gain_block_steps(dm);
  io.pm = post_mean;
  io.pP = post_cov;
  io.smean = smooth_mean;
  io.scov = smooth_cov;
  io.scross = smooth_cross;
  hipStream_t st = (hipStream_t)stream;
  const StHyp hy = make_hyp(hyp);
  BN_TIMED(KID_ST_SMOOTHER, st);
  return dm.KT == 1 ? launch_st_smoother<1>(st, dm, hy, dt, aq, filter_mean, filter_cov, io)
                    : launch_st_smoother<2>(st, dm, hy, dt, aq, filter_mean, filter_cov, io);
}

int bn_st_marginals(const bn_st_dims* dims, const double* B, const double* cdiag, const double* post_mean,
                    const double* post_cov, double* mean_f, double* var_f, void* stream) {
  StDims dm;
  if (int rc = check_dims(dims, dm)) return rc;
  if (!B || !cdiag || !post_mean || !post_cov || !mean_f || !var_f)
    return st_fail(BN_EINVAL, "NULL argument to bn_st_marginals");
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(k_st_marginals, dim3(dm.T, dm.K), dim3(kT), 0, st, dm, B, cdiag, post_mean, post_cov, mean_f,
                     var_f);
  ST_HIP_CHECK(hipGetLastError());
  return BN_OK;
}

int bn_st_sum(int32_t n_runs, int32_t n_steps, const double* per_step, double* per_run, void* stream) {
  if (n_runs < 1 || n_steps < 1 || !per_step || !per_run) return st_fail(BN_EINVAL, "bad argument to bn_st_sum");
  hipStream_t st = (hipStream_t)stream;
  BN_TIMED(KID_ST_SUM, st);
  hipLaunchKernelGGL(k_st_sum, dim3(n_runs), dim3(kT), 0, st, n_steps, per_step, per_run);
  ST_HIP_CHECK(hipGetLastError());
  return BN_OK;
}

int64_t bn_mf_workspace_bytes(const bn_st_dims* dims) {
  StDims dm;
  if (check_dims(dims, dm) != BN_OK) return -1;
  return 2 * (int64_t)dm.K * dm.T * dm.M * (int64_t)sizeof(double) + 256;
}

int bn_mf_pseudo(const bn_st_dims* dims, const double* Lw, const double* zw, double* noise, double* y,
                 void* stream) {
  StDims dm;
  if (int rc = check_dims(dims, dm)) return rc;
  if (!Lw || !zw || !noise || !y) return st_fail(BN_EINVAL, "NULL argument to bn_mf_pseudo");
  if (int rc = set_smem_limits()) return rc;
  hipStream_t st = (hipStream_t)stream;
  BN_TIMED(KID_MF_PSEUDO, st);
  hipLaunchKernelGGL(k_mf_pseudo, dim3(dm.T, dm.K), dim3(kT), kPseudoSmem, st, dm, Lw, zw, noise, y);
  ST_HIP_CHECK(hipGetLastError());
  return BN_OK;
}

int bn_mf_filter(const bn_st_dims* dims, const bn_st_hypers* hyp, int32_t parallel, const double* dt,
                 const double* y, const double* noise, double* filter_mean, double* filter_cov, double* ell_steps,
                 double* loglik, void* workspace, void* stream) {
  StDims dm;
  if (int rc = check_dims(dims, dm)) return rc;
  if (!hyp || !dt || !y || !noise || !filter_mean || !filter_cov || !ell_steps || !loglik)
    return st_fail(BN_EINVAL, "NULL argument to bn_mf_filter");
  if (parallel && !workspace) return st_fail(BN_EINVAL, "the associative form needs bn_mf_workspace_bytes of workspace");
  double* ws = (double*)workspace;
  const int64_t ktm = (int64_t)dm.K * dm.T * dm.M;
  MfFilterIO io{dt, y, noise, filter_mean, filter_cov, ell_steps, ws, ws ? ws + ktm : nullptr};
  const StHyp hy = make_hyp(hyp);
  hipStream_t st = (hipStream_t)stream;
  if (!parallel) {
    BN_TIMED(KID_MF_FILTER, st);
    if (dm.KT == 1) hipLaunchKernelGGL(k_mf_filter<1>, dim3(dm.K), dim3(kT), 0, st, dm, hy, io);
    else hipLaunchKernelGGL(k_mf_filter<2>, dim3(dm.K), dim3(kT), 0, st, dm, hy, io);
    ST_HIP_CHECK(hipGetLastError());
  } else {
    const dim3 grid(dm.T, dm.K);
    const int lanes = mf_lanes(dm);
    const int nb = (int)((dm.K * (int64_t)dm.M + lanes - 1) / lanes);
    const size_t lds = mf_table_doubles(dm) * 8;
    {
      BN_TIMED(KID_MF_SDIAG, st);
      if (dm.KT == 1) hipLaunchKernelGGL((k_mf_sdiag<1, false>), grid, dim3(kT), 0, st, dm, hy, io);
      else hipLaunchKernelGGL((k_mf_sdiag<2, false>), grid, dim3(kT), 0, st, dm, hy, io);
      ST_HIP_CHECK(hipGetLastError());
    }
    {
      BN_TIMED(KID_MF_BLOCKS, st);
      if (dm.KT == 1) hipLaunchKernelGGL(k_mf_blocks<1>, dim3(nb), dim3(kMfBlocksT), lds, st, dm, hy, io, lanes);
      else hipLaunchKernelGGL(k_mf_blocks<2>, dim3(nb), dim3(kMfBlocksT), lds, st, dm, hy, io, lanes);
      ST_HIP_CHECK(hipGetLastError());
    }
    {
      BN_TIMED(KID_MF_SDIAG, st);
      if (dm.KT == 1) hipLaunchKernelGGL((k_mf_sdiag<1, true>), grid, dim3(kT), 0, st, dm, hy, io);
      else hipLaunchKernelGGL((k_mf_sdiag<2, true>), grid, dim3(kT), 0, st, dm, hy, io);
      ST_HIP_CHECK(hipGetLastError());
    }
  }
  {
    BN_TIMED(KID_ST_SUM, st);
    hipLaunchKernelGGL(k_st_sum, dim3(dm.K), dim3(kT), 0, st, dm.T, ell_steps, loglik);
  }
  ST_HIP_CHECK(hipGetLastError());
  return BN_OK;
}

int bn_mf_smoother(const bn_st_dims* dims, const bn_st_hypers* hyp, const double* dt, const double* filter_mean,
                   const double* filter_cov, double* post_mean, double* post_var, int64_t var_step_stride,
                   int64_t var_elem_stride, double* smooth_mean, double* smooth_cov, double* gains, void* stream) {
  StDims dm;
  if (int rc = check_dims(dims, dm)) return rc;
  if (!hyp || !dt || !filter_mean || !filter_cov) return st_fail(BN_EINVAL, "NULL argument to bn_mf_smoother");
  if (!post_mean && !post_var && !smooth_mean && !smooth_cov && !gains)
    return st_fail(BN_EINVAL, "bn_mf_smoother: no output requested");
  if (post_var && (var_step_stride < 0 || var_elem_stride < 0 ||
                   (dm.M - 1) * var_elem_stride >= (var_step_stride > 0 ? var_step_stride : INT64_MAX)))
    return st_fail(BN_EINVAL, "bn_mf_smoother: post_var strides overlap");
  MfSmootherIO io{dt, filter_mean, filter_cov, post_mean, post_var, var_step_stride, var_elem_stride,
                  smooth_mean, smooth_cov, gains};
  hipStream_t st = (hipStream_t)stream;
  const int lanes = mf_lanes(dm);
  const int nb = (int)((dm.K * (int64_t)dm.M + lanes - 1) / lanes);
  const size_t lds =
      (mf_table_doubles(dm) + (size_t)2 * kMfTile * (dm.KT == 1 ? kMfFields<1> : kMfFields<2>) * 64) * 8;
  if (int rc = set_smem_limits()) return rc;
  BN_TIMED(KID_MF_SMOOTHER, st);
  if (dm.KT == 1) hipLaunchKernelGGL(k_mf_smoother<1>, dim3(nb), dim3(kMfSmootherT), lds, st, dm, make_hyp(hyp), io, lanes);
  else hipLaunchKernelGGL(k_mf_smoother<2>, dim3(nb), dim3(kMfSmootherT), lds, st, dm, make_hyp(hyp), io, lanes);
  ST_HIP_CHECK(hipGetLastError());
  return BN_OK;
}

int64_t bn_ih_workspace_bytes(const bn_st_dims* dims, int32_t heteroscedastic) {
  StDims dm;
  if (check_dims(dims, dm) != BN_OK) return -1;
  const int64_t K = dm.K, M = dm.M, T = dm.T;
  int64_t n = ih_head(dm) + K * M * M + K + K * kTiedParts * M * M;
  if (heteroscedastic) n += K * T * M * M + K * T;
  return n * (int64_t)sizeof(double) + 256;
}

int bn_ih_tied(const bn_st_dims* dims, const double* Lw, double* noise_tied, void* workspace, void* stream) {
  StDims dm;
  if (int rc = check_dims(dims, dm)) return rc;
  if (!Lw || !noise_tied || !workspace) return st_fail(BN_EINVAL, "NULL argument to bn_ih_tied");
  // partial sums after bn_ih_filter's regions (see bn_ih_workspace_bytes)
  const int64_t K = dm.K, M = dm.M;
  double* part = (double*)workspace + ih_head(dm) + K * M * M + K;
  hipStream_t st = (hipStream_t)stream;
  BN_TIMED(KID_IH_TIED, st);
  hipLaunchKernelGGL(k_ih_tied_part, dim3(kTiedParts, dm.K), dim3(kT), kTiedSmem, st, dm, Lw, part);
  ST_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(k_ih_tied, dim3(dm.K), dim3(kT), 0, st, dm, part, noise_tied);
  ST_HIP_CHECK(hipGetLastError());
  return BN_OK;
}

int bn_ih_filter(const bn_st_dims* dims, const bn_st_hypers* hyp, const double* step, int32_t iters,
                 int32_t heteroscedastic, const double* y, const double* noise, const double* noise_tied, double* dare,
                 double* filter_cov, double* filter_mean, double* ell_steps, double* loglik, void* workspace,
                 void* stream) {
  StDims dm;
  if (int rc = check_dims(dims, dm)) return rc;
  if (!hyp || !step || !y || !noise_tied || !dare || !filter_cov || !filter_mean || !ell_steps || !loglik ||
      !workspace || (heteroscedastic && !noise))
    return st_fail(BN_EINVAL, "NULL argument to bn_ih_filter");
  if (iters < 0) return st_fail(BN_EINVAL, "bn_ih_filter: iters must be >= 0");
  if (int rc = set_smem_limits()) return rc;
  const int64_t K = dm.K, M = dm.M;
  double* ws = (double*)workspace;
  IhIO io{};
  io.aq = ws;
  io.y = y;
  io.R = noise;
  io.Rt = noise_tied;
  io.X = dare;
  io.cov = filter_cov;
  io.STn = ws + ih_head(dm);
  io.ldT = io.STn + K * M * M;
  io.Sn = heteroscedastic ? io.ldT + K + K * kTiedParts * M * M : nullptr;
  io.ldS = heteroscedastic ? io.Sn + K * dm.T * M * M : nullptr;
  io.fmean = filter_mean;
  io.ell = ell_steps;
  io.iters = iters;
  io.hetero = heteroscedastic ? 1 : 0;
  const StHyp hy = make_hyp(hyp);
  hipStream_t st = (hipStream_t)stream;
  {
    BN_TIMED(KID_IH_DARE, st);
    launch_ih_transitions(st, dm, hy, step, ws);
    if (dm.KT == 1) launch_ih_dare<1>(st, dm, io);
    else launch_ih_dare<2>(st, dm, io);
    ST_HIP_CHECK(hipGetLastError());
  }
  {
    BN_TIMED(KID_IH_SINV, st);
    if (heteroscedastic) hipLaunchKernelGGL(k_ih_sinv<false>, dim3(dm.T, dm.K), dim3(kT), 0, st, dm, io);
    else hipLaunchKernelGGL(k_ih_sinv<true>, dim3(1, dm.K), dim3(kT), 0, st, dm, io);
    ST_HIP_CHECK(hipGetLastError());
  }
  {
    BN_TIMED(KID_IH_FILTER, st);
    if (dm.KT == 1) {
      hipLaunchKernelGGL(k_ih_filter<1>, dim3(dm.K), dim3(8 * kMaxM), 0, st, dm, io);
      hipLaunchKernelGGL(k_ih_ell<1>, dim3(dm.T, dm.K), dim3(64), 0, st, dm, io);
    } else {
      hipLaunchKernelGGL(k_ih_filter<2>, dim3(dm.K), dim3(8 * kMaxM), 0, st, dm, io);
      hipLaunchKernelGGL(k_ih_ell<2>, dim3(dm.T, dm.K), dim3(64), 0, st, dm, io);
    }
    ST_HIP_CHECK(hipGetLastError());
  }
  {
    BN_TIMED(KID_ST_SUM, st);
    hipLaunchKernelGGL(k_st_sum, dim3(dm.K), dim3(kT), 0, st, dm.T, ell_steps, loglik);
  }
  ST_HIP_CHECK(hipGetLastError());
  return BN_OK;
}

int bn_ih_smoother(const bn_st_dims* dims, const bn_st_hypers* hyp, const double* step, int32_t iters,
                   const double* filter_mean, const double* dare, const double* filter_cov, double* dare_smoother,
                   double* gain, double* post_mean, double* post_cov, double* smooth_mean, void* workspace,
                   void* stream) {
  StDims dm;
  if (int rc = check_dims(dims, dm)) return rc;
  if (!hyp || !step || !filter_mean || !dare || !filter_cov || !dare_smoother || !workspace)
    return st_fail(BN_EINVAL, "NULL argument to bn_ih_smoother");
  if (iters < 0) return st_fail(BN_EINVAL, "bn_ih_smoother: iters must be >= 0");
  if (int rc = set_smem_limits()) return rc;
  const int64_t K = dm.K;
  double* ws = (double*)workspace;
  double* rec = ws + K * 2 * dm.KT * dm.KT;
  double* G = gain ? gain : rec + K * map_doubles(dm);
  const StGainIO gi{ws, nullptr, filter_cov, rec, 0, 1, dare, G};
  StSmootherIO si{};
  si.rec = rec;
  si.tb = 1;
  si.xs = dare_smoother;
  si.iters = iters;
  const IhSmIO io{ws, filter_mean, dare_smoother, G, post_mean, post_cov, smooth_mean};
  const StHyp hy = make_hyp(hyp);
  hipStream_t st = (hipStream_t)stream;
  BN_TIMED(KID_IH_SMOOTHER, st);
  launch_ih_transitions(st, dm, hy, step, ws);
  if (dm.KT == 1) {
    launch_ih_smoother<1>(st, dm, gi, si);
    hipLaunchKernelGGL(k_ih_means<1>, dim3(dm.K), dim3(4 * kMaxD), 0, st, dm, io);
  } else {
    launch_ih_smoother<2>(st, dm, gi, si);
    hipLaunchKernelGGL(k_ih_means<2>, dim3(dm.K), dim3(4 * kMaxD), 0, st, dm, io);
  }
  if (post_cov) hipLaunchKernelGGL(k_ih_spread, dim3(dm.T, dm.K), dim3(kT), 0, st, dm, io);
  ST_HIP_CHECK(hipGetLastError());
  return BN_OK;
}

int bn_st_predict(const bn_st_dims* dims, const bn_st_hypers* hyp, const double* t_train, int32_t n_test,
                  int32_t n_loc_test, const double* t_test, const double* B_test, const double* cdiag_test,
                  const double* smooth_mean, const double* smooth_cov, const double* smooth_cross,
                  const double* steady_cov, double* mean, double* var, void* stream) {
  StDims dm;
  if (int rc = check_dims(dims, dm)) return rc;
  if (!hyp || !t_train || !t_test || !B_test || !cdiag_test || !smooth_mean || !mean || !var ||
      (!steady_cov && (!smooth_cov || !smooth_cross)))
    return st_fail(BN_EINVAL, "NULL argument to bn_st_predict");
  if (n_test < 1 || n_loc_test < 1) return st_fail(BN_EINVAL, "bn_st_predict: empty test set");
  StPredIO io{t_train, t_test, B_test, cdiag_test, smooth_mean, smooth_cov, smooth_cross, steady_cov, mean, var, n_test,
              n_loc_test};
  hipStream_t st = (hipStream_t)stream;
  if (dm.KT == 1)
    hipLaunchKernelGGL(k_st_predict<1>, dim3(n_test, dm.K), dim3(kT), 0, st, dm, make_hyp(hyp), io);
  else
    hipLaunchKernelGGL(k_st_predict<2>, dim3(n_test, dm.K), dim3(kT), 0, st, dm, make_hyp(hyp), io);
  ST_HIP_CHECK(hipGetLastError());
  return BN_OK;
}

}  // extern "C"
