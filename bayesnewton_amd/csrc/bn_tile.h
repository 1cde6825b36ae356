// FP64 matrix-core tile primitives of the space-time kernels: 16 x 16 tiles held by one
// wavefront, operands in LDS, and the Cholesky factor of a 16 x 16 block with its inverse.
//
// v_mfma_f64_16x16x4f64 takes A[l%16][k + l/16] and B[k + l/16][l%16] from lane l and
// returns, in result register q, element (l/16 + 4q, l%16).  An LDS matrix is stored row by
// row with a stride of 16 n + 2 doubles: a fragment read with the row on l%16 then covers
// every bank once per half-wavefront (stride = 4 times an odd number of 32-bit words), and
// since B[k][j] = X'[k][j] = X[j][k] has that form too, products A X' need no transposed copy.
#pragma once
#include <hip/hip_runtime.h>

namespace bn {

typedef double tile4 __attribute__((ext_vector_type(4)));

__device__ inline tile4 tile_zero() { return tile4{0.0, 0.0, 0.0, 0.0}; }

__device__ inline tile4 mfma16(double a, double b, tile4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Orders the LDS accesses of one wavefront's lanes (the hardware runs them in order; this
// keeps the compiler from moving them).
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Values the compiler must take as new here.  Lane and wavefront numbers go through these at
// the start of a phase of a long kernel, so that the address arithmetic of the phase is done
// there instead of being hoisted out of the step loop into registers that the tiles need.
__device__ inline int fresh_v(int x) {
  asm volatile("" : "+v"(x));
  return x;
}
__device__ inline int fresh_s(int x) {
  asm volatile("" : "+s"(x));
  return x;
}

// fragment with the row on l%16: X[r0 + l%16][k0 + l/16]
__device__ inline double frag(const double* X, int ld, int r0, int k0, int l) {
  return X[(r0 + (l & 15)) * ld + k0 + (l >> 4)];
}

// fragment with the row on l/16: X[k0 + l/16][c0 + l%16]
__device__ inline double frag_t(const double* X, int ld, int k0, int c0, int l) {
  return X[(k0 + (l >> 4)) * ld + c0 + (l & 15)];
}

__device__ inline void tile_store(double* X, int ld, int r0, int c0, tile4 v, int l) {
  double* p = X + (r0 + (l >> 4)) * ld + c0 + (l & 15);
#pragma unroll
  for (int q = 0; q < 4; ++q) p[4 * q * ld] = v[q];
}

// the transpose of the tile
__device__ inline void tile_store_t(double* X, int ld, int r0, int c0, tile4 v, int l) {
  double* p = X + (r0 + (l & 15)) * ld + c0 + (l >> 4);
#pragma unroll
  for (int q = 0; q < 4; ++q) p[4 * q] = v[q];
}

// sign times the four fragments of columns k0 .. k0 + 15
__device__ inline void frag4(double (&a)[4], const double* X, int ld, int r0, int k0, double sign, int l) {
#pragma unroll
  for (int c = 0; c < 4; ++c) a[c] = sign * frag(X, ld, r0, k0 + 4 * c, l);
}

// c += A B' over one 16-wide block of the inner dimension: A rows r0.., B rows j0.., columns k0..
__device__ inline tile4 tile_mul_t(const double* A, int lda, int r0, const double* B, int ldb, int j0, int ka, int kb,
                                   tile4 c, int l) {
#pragma unroll
  for (int kk = 0; kk < 16; kk += 4) c = mfma16(frag(A, lda, r0, ka + kk, l), frag(B, ldb, j0, kb + kk, l), c);
  return c;
}

__device__ inline double lane_bcast(double v, int lane) {
  const int lo = __builtin_amdgcn_readlane((int)__double_as_longlong(v), lane);
  const int hi = __builtin_amdgcn_readlane((int)(__double_as_longlong(v) >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

constexpr int kDiagLd = 18;  // row stride of a 16 x 16 block on its own in LDS

// Cholesky factor of a 16 x 16 symmetric positive definite block and its inverse, by one
// wavefront.  Lanes 0-15 start with the rows of A, the others with the columns of I; the
// elimination step of pivot k, w_j -= l_jk w_k / sqrt(d), is the same instruction for both
// (a Cholesky update of row r, a forward substitution of column c), with l_jk broadcast to
// every lane through a scalar register.  16 pivots deep and latency bound.
//   D (LDS, row stride ld): A in (A's rows; only the lower triangle is read for the factor),
//   L^-1 out (rows, zero above the diagonal).
//   L (optional, row stride ldl): the factor, zero above the diagonal.  Row tiles below the block
//   get their factors as tile * L^-T.
// A non-positive pivot gives NaN, which propagates.
// The scaling by 1 / sqrt(d) is the hardware estimate y and one third-order Newton step,
// folded into the scaled column: w (y + y e (1/2 + 3/8 e)), e = 1 - d y^2.
// Raised wave priority: the pivot chain competes for the FP64 pipe with the matrix
// instructions of the wavefronts on the same SIMD, each of which holds it for 64 cycles.
template <bool KEEP = false>
__device__ inline void chol16_inverse(double* D, int ld, int l, double* L = nullptr, int ldl = 0) {
  const int r = l & 15;
  double w[16];
  __builtin_amdgcn_s_setprio(3);
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const double a = D[r * ld + j];
    w[j] = l < 16 ? a : (j == r ? 1.0 : 0.0);
  }
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const double d = lane_bcast(w[k], k);
    const double y = __builtin_amdgcn_rsq(d), wy = w[k] * y;
    const double e = fma(-d * y, y, 1.0), p = fma(0.375, e, 0.5);
    const double m = fma(wy * e, p, wy);
    w[k] = m;
#pragma unroll
    for (int j = k + 1; j < 16; ++j) w[j] = fma(-lane_bcast(m, j), m, w[j]);
  }
  wave_sync();
  if (l >= 16 && l < 32) {
#pragma unroll
    for (int j = 0; j < 16; ++j) D[j * ld + r] = w[j];  // column r of L^-1: zero above the diagonal
  }
  if (KEEP && l < 16) {
#pragma unroll
    for (int j = 0; j < 16; ++j) L[r * ldl + j] = j <= r ? w[j] : 0.0;
  }
  __builtin_amdgcn_s_setprio(0);
}

// A tile in memory: four consecutive doubles a lane (no alignment beyond a double's is assumed).
typedef double tile4_mem __attribute__((ext_vector_type(4), aligned(8)));
__device__ inline tile4 tile_get(const double* p, int l) { return *reinterpret_cast<const tile4_mem*>(p + 4 * l); }
__device__ inline void tile_put(double* p, tile4 v, int l) { *reinterpret_cast<tile4_mem*>(p + 4 * l) = v; }

}  // namespace bn
