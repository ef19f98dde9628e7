// PCA fit on the GPU: FP64 mean and covariance of the base, symmetric
// eigen-decomposition on the host (Householder + QL, FP64), eigenvectors sorted
// by descending eigenvalue with a deterministic sign (largest-magnitude
// component positive).  Replaces the reference's Eigen-based PCA::PCA
// (pca.cpp:4-58: mean, covariance / (n - 1), SelfAdjointEigenSolver, columns
// reordered by descending eigenvalue), which holds the whole base as doubles
// on the host (pca.h:15-21).
//
// Two passes over the base.  Column sums: rows split over workgroups, the
// per-workgroup partials summed in a fixed order.  Covariance: the d x d
// result is cut into 128 x 128 tiles; a workgroup accumulates, for one tile
// on or above the diagonal and one range of rows, sum (x - mu)_i (x - mu)_j
// in FP64 matrix instructions, the centred rows staged through LDS 32 at a
// time; the per-row-range partials are again summed in a fixed order and what
// lies below the diagonal is the mirror image (the products are the same
// numbers in the same order, so C is exactly symmetric).  Everything is
// deterministic.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <numeric>
#include <vector>

#include "ctx.h"

namespace rte {

constexpr int kPcaTile = 128;
constexpr int kPcaMaxD = 4096;

// Sum of x[0], x[step], ... (n of them) in order: the loads of kSumAhead
// elements are issued together, so the chain of additions and one memory round
// trip per kSumAhead elements are what it takes (one round trip per element
// otherwise: 1M x 128 column sums 808 -> 100 us, the reductions of their and
// the covariance's partials 118 -> 13 and 123 -> 25 us).
constexpr int kSumAhead = 32;
template <typename T>
__device__ __forceinline__ double ordered_sum(const T* __restrict__ x, int64_t step, int64_t n) {
  double s = 0.0;
  int64_t r = 0;
  for (; r + kSumAhead <= n; r += kSumAhead) {
    T v[kSumAhead];
#pragma unroll
    for (int i = 0; i < kSumAhead; ++i) v[i] = x[(r + i) * step];
#pragma unroll
    for (int i = 0; i < kSumAhead; ++i) s += (double)v[i];
  }
  for (; r < n; ++r) s += (double)x[r * step];
  return s;
}

__global__ __launch_bounds__(256) void col_sum_kernel(const float* __restrict__ X, int64_t n,
                                                      int d, int64_t stride, int64_t rpb,
                                                      double* __restrict__ partial) {
  const int64_t r0 = (int64_t)blockIdx.x * rpb;
  const int64_t r1 = r0 + rpb < n ? r0 + rpb : n;
  for (int c = threadIdx.x; c < d; c += blockDim.x)
    partial[(int64_t)blockIdx.x * d + c] = ordered_sum(X + r0 * stride + c, stride, r1 - r0);
}

__global__ void col_mean_kernel(const double* __restrict__ partial, int nb, int d, int64_t n,
                                double* __restrict__ mean) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d) return;
  mean[c] = ordered_sum(partial + c, d, nb) / (double)n;
}

// grid (row ranges, tile pairs); tile pair p -> (bi, bj), bi <= bj, row-major
// over the upper triangle of the nt x nt tile grid.
//
// Products on v_mfma_f64_16x16x4: lane l gives A[l % 16][l / 16] and
// B[l / 16][l % 16] and holds D[4 r + l / 16][l % 16], and an element is the
// chain of four FMAs in ascending k, so a sum has the bits of one FMA per row,
// row after row.  (The FP64 vector unit has the same rate, but an 8 x 8 block a
// thread reads 128 bytes of LDS per 64 FMAs, which takes LDS as long as the
// FMAs take.)  Both operands of a block of 16 columns are the same 64 numbers.
// Off the diagonal a wave has 4 x 4 blocks of 16 x 16.  On it only the 36 blocks
// with row <= column are computed, nine a wave: block rows w and 7 - w.  A row
// of LDS is 144 doubles, so the four rows of an operand lie in both halves of
// the banks.  The next rows' loads are in flight during the products.
// 1M x 128: 420 us, 1225 us with an 8 x 8 block a thread.
constexpr int kCovRows = 32;
constexpr int kCovPitch = kPcaTile + 16;
typedef double f64x4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256, 2) void cov_partial_kernel(const float* __restrict__ X, int64_t n,
                                                          int d, int64_t stride,
                                                          const double* __restrict__ mean,
                                                          int64_t rpb, int nt,
                                                          double* __restrict__ partial) {
  __shared__ double ra[kCovRows * kCovPitch];
  __shared__ double rb[kCovRows * kCovPitch];
  int p = blockIdx.y, bi = 0;
  while (p >= nt - bi) {
    p -= nt - bi;
    ++bi;
  }
  const int bj = bi + p;
  const int c0 = bi * kPcaTile, c1 = bj * kPcaTile;
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t r0 = (int64_t)blockIdx.x * rpb;
  const int64_t r1 = r0 + rpb < n ? r0 + rpb : n;
  // thread t stages column t % 128 of rows t / 128 + 2 i; rows past the range
  // are zeros, columns past d (any valid one) only reach elements past d
  constexpr int kPer = kCovRows * kPcaTile / 256;
  const int sc = t & (kPcaTile - 1), sr = t / kPcaTile;
  const int ca = min(c0 + sc, d - 1), cb = min(c1 + sc, d - 1);
  const double ma = mean[ca], mb = mean[cb];
  auto load = [&](int64_t rs, int c, float (&v)[kPer]) {  // at clamped, valid addresses
#pragma unroll
    for (int i = 0; i < kPer; ++i) v[i] = X[min(rs + sr + 2 * i, n - 1) * stride + c];
  };
  auto stage = [&](int64_t rs, const float (&v)[kPer], double m, double* dst) {
    dst += sr * kCovPitch + sc;
    if (rs + kCovRows <= r1) {
#pragma unroll
      for (int i = 0; i < kPer; ++i) dst[2 * i * kCovPitch] = (double)v[i] - m;
    } else {
#pragma unroll
      for (int i = 0; i < kPer; ++i)
        dst[2 * i * kCovPitch] = rs + sr + 2 * i < r1 ? (double)v[i] - m : 0.0;
    }
  };
  double* out = partial + (int64_t)blockIdx.x * d * d;
  const int lo = (lane >> 4) * kCovPitch + (lane & 15);  // the lane's element of an operand
  auto store = [&](int gi, int gj, const f64x4& v) {     // a 16 x 16 block at (gi, gj)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = gi + 4 * r + (lane >> 4), j = gj + (lane & 15);
      if (i < d && j < d) out[(int64_t)i * d + j] = v[r];
    }
  };
  if (bi == bj) {
    constexpr int kT = 9;
    f64x4 acc[kT];
    int br[kT], bc[kT];  // block row and column of the wave's blocks
#pragma unroll
    for (int q = 0; q < kT; ++q) {
      acc[q] = f64x4{0.0, 0.0, 0.0, 0.0};
      br[q] = q < 8 - w ? w : 7 - w;
      bc[q] = q < 8 - w ? w + q : q - 1;
    }
    float va[kPer];
    if (r0 < r1) load(r0, ca, va);
    for (int64_t rs = r0; rs < r1; rs += kCovRows) {
      stage(rs, va, ma, ra);
      __syncthreads();
      if (rs + kCovRows < r1) load(rs + kCovRows, ca, va);
#pragma unroll 2
      for (int k = 0; k < kCovRows; k += 4) {
        double fa[kT], fb[kT];
#pragma unroll
        for (int q = 0; q < kT; ++q) {
          fa[q] = ra[k * kCovPitch + 16 * br[q] + lo];
          fb[q] = ra[k * kCovPitch + 16 * bc[q] + lo];
        }
#pragma unroll
        for (int q = 0; q < kT; ++q)
          acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[q], fb[q], acc[q], 0, 0, 0);
      }
      __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < kT; ++q) store(c0 + 16 * br[q], c1 + 16 * bc[q], acc[q]);
  } else {
    const int wi = 4 * (w >> 1), wj = 4 * (w & 1);
    f64x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
    float va[kPer], vb[kPer];
    if (r0 < r1) {
      load(r0, ca, va);
      load(r0, cb, vb);
    }
    for (int64_t rs = r0; rs < r1; rs += kCovRows) {
      stage(rs, va, ma, ra);
      stage(rs, vb, mb, rb);
      __syncthreads();
      if (rs + kCovRows < r1) {
        load(rs + kCovRows, ca, va);
        load(rs + kCovRows, cb, vb);
      }
#pragma unroll 2
      for (int k = 0; k < kCovRows; k += 4) {
        double fa[4], fb[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          fa[q] = ra[k * kCovPitch + 16 * (wi + q) + lo];
          fb[q] = rb[k * kCovPitch + 16 * (wj + q) + lo];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[i], fb[j], acc[i][j], 0, 0, 0);
      }
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) store(c0 + 16 * (wi + i), c1 + 16 * (wj + j), acc[i][j]);
  }
}

__global__ void cov_reduce_kernel(const double* __restrict__ partial, int nb, int d, int64_t n,
                                  double* __restrict__ C) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)d * d) return;
  const int i = (int)(e / d), j = (int)(e - (int64_t)i * d);
  if (i / 16 > j / 16) return;  // blocks below the diagonal: mirror images
  const double v =
      ordered_sum(partial + e, (int64_t)d * d, nb) / (double)(n > 1 ? n - 1 : 1);  // pca.cpp:8-9
  C[e] = v;
  if (i / 16 < j / 16) C[(int64_t)j * d + i] = v;
}

// out[i][c] = sum_j ((double)X[i][j] - (double)mu[j]) * (double)R[j][c],
// j ascending, multiply then add (the library is built without contraction),
// stored FP32 -- the FP64 rotation of pca.cpp:122-139.
//
// Bound by the FP64 multiplies and adds (no FMA, so no matrix instruction: its
// products are not rounded).  A lane has one row and 16 columns, a wave 64 rows:
// the centred values, staged through LDS as [j][row] 64 columns of X at a time,
// cost one 8-byte read per 32 operations, and R, widened to FP64 in rows of a
// multiple of 16 columns, comes by scalar loads.  A workgroup has up to eight
// waves, 128 columns.  1M x 128 x 128: 1275 us (834 us at the nominal rate);
// 1728 us with eight rows and one column a thread, whose reads of the centred
// values took LDS twice as long as the arithmetic.
constexpr int kRotRows = 64;
constexpr int kRotCols = 16;
constexpr int kRotK = 64;
__global__ __launch_bounds__(256) void widen_kernel(const float* __restrict__ R, int d, int d_out,
                                                    int ldr, double* __restrict__ W) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= (int64_t)(d + 1) * ldr) return;
  const int j = (int)(e / ldr), c = (int)(e - (int64_t)j * ldr);
  W[e] = j < d && c < d_out ? (double)R[(int64_t)j * d_out + c] : 0.0;
}

__global__ __launch_bounds__(512) void pca_rotate_kernel(const float* __restrict__ X, int64_t n,
                                                         int d, int64_t stride,
                                                         const double* __restrict__ W, int ldr,
                                                         const float* __restrict__ mu, int d_out,
                                                         float* __restrict__ out) {
  constexpr int kPitch = kRotRows + 1;
  __shared__ double xs[(kRotK + 1) * kPitch];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6), nw = blockDim.x >> 6;
  const int c0 = blockIdx.y * kPcaTile + w * kRotCols;
  const bool active = c0 < d_out;
  const int64_t row0 = (int64_t)blockIdx.x * kRotRows;
  double acc[kRotCols];
#pragma unroll
  for (int i = 0; i < kRotCols; ++i) acc[i] = 0.0;
  typedef const __attribute__((address_space(4))) double* cptr;  // read-only: scalar loads
  const cptr Wc = (cptr)W + c0;
  for (int j0 = 0; j0 < d; j0 += kRotK) {
    const int jn = d - j0 < kRotK ? d - j0 : kRotK;
    // wave w stages rows w, w + nw, ...; a lane its column (past d: not used)
    const int j = min(j0 + lane, d - 1);
    const double m = (double)mu[j];
#pragma unroll 8
    for (int r = w; r < kRotRows; r += nw)
      xs[lane * kPitch + r] = (double)X[min(row0 + r, n - 1) * stride + j] - m;
    __syncthreads();
    if (active) {
      double r[kRotCols], x = xs[lane];
      cptr wr = Wc + (int64_t)j0 * ldr;
#pragma unroll
      for (int i = 0; i < kRotCols; ++i) r[i] = wr[i];
#pragma unroll 2
      for (int k = 0; k < jn; ++k) {
        // scalar loads return in any order: wait for this row's, ask for the
        // next (W and xs have a spare one), then multiply
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        __builtin_amdgcn_sched_barrier(0);
        wr += ldr;
        double rn[kRotCols];
        const double xn = xs[(k + 1) * kPitch + lane];
#pragma unroll
        for (int i = 0; i < kRotCols; ++i) rn[i] = wr[i];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kRotCols; ++i) acc[i] = acc[i] + x * r[i];
        x = xn;
#pragma unroll
        for (int i = 0; i < kRotCols; ++i) r[i] = rn[i];
      }
    }
    __syncthreads();
  }
  const int64_t row = row0 + lane;
  if (active && row < n) {
    float* o = out + row * d_out + c0;
    if (c0 + kRotCols <= d_out && (d_out & 3) == 0 && ((uintptr_t)out & 15) == 0) {
#pragma unroll
      for (int i = 0; i < kRotCols; i += 4)
        *reinterpret_cast<float4*>(o + i) =
            make_float4((float)acc[i], (float)acc[i + 1], (float)acc[i + 2], (float)acc[i + 3]);
    } else {
#pragma unroll
      for (int i = 0; i < kRotCols; ++i)
        if (c0 + i < d_out) o[i] = (float)acc[i];
    }
  }
}

// The same for few columns, four or eight a wave: all four waves stage the rows, the
// next 64 columns of X on their way during the products, and R's come from LDS,
// widened there, so one launch does it.  The kernel above has a wave or two a
// workgroup here, which stage 64 rows alone and wait for scalar loads at every column
// of X.  Bound by the launch and a few round trips at 1000 x 128 to 3 columns (34 us
// with both copies to the device, 70 with the kernel above), by memory and LDS (three
// reads for 8 operations a wave) at 1M x 96 to 3: 174 us, 2.3 TB/s.
template <int C>  // columns a wave
__global__ __launch_bounds__(256) void pca_rotate_narrow_kernel(
    const float* __restrict__ X, int64_t n, int d, int64_t stride, const float* __restrict__ R,
    const float* __restrict__ mu, int d_out, float* __restrict__ out) {
  constexpr int kPitch = kRotRows + 1, kPer = kRotRows / 4, kCols = 4 * C;
  __shared__ double xs[kRotK * kPitch];
  __shared__ __attribute__((aligned(16))) double rs[kRotK * kCols];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6), c0 = C * w;
  const int64_t row0 = (int64_t)blockIdx.x * kRotRows;
  double acc[C];
#pragma unroll
  for (int i = 0; i < C; ++i) acc[i] = 0.0;
  float v[kPer];
  auto load = [&](int j0) {  // at clamped, valid addresses
    const int j = min(j0 + lane, d - 1);
#pragma unroll
    for (int i = 0; i < kPer; ++i) v[i] = X[min(row0 + w + 4 * i, n - 1) * stride + j];
  };
  load(0);
  for (int j0 = 0; j0 < d; j0 += kRotK) {
    const int jn = d - j0 < kRotK ? d - j0 : kRotK;
    const double m = (double)mu[min(j0 + lane, d - 1)];
#pragma unroll
    for (int i = 0; i < kPer; ++i) xs[lane * kPitch + w + 4 * i] = (double)v[i] - m;
    for (int e = t; e < kRotK * kCols; e += 256) {
      const int k = e / kCols, c = e % kCols;
      rs[e] = k < jn && c < d_out ? (double)R[(int64_t)(j0 + k) * d_out + c] : 0.0;
    }
    __syncthreads();
    if (j0 + kRotK < d) load(j0 + kRotK);
    if (c0 < d_out) {
#pragma unroll 8
      for (int k = 0; k < jn; ++k) {
        const double x = xs[k * kPitch + lane];
#pragma unroll
        for (int i = 0; i < C; ++i) acc[i] = acc[i] + x * rs[k * kCols + c0 + i];
      }
    }
    __syncthreads();
  }
  const int64_t row = row0 + lane;
  if (row < n)
#pragma unroll
    for (int i = 0; i < C; ++i)
      if (c0 + i < d_out) out[row * d_out + c0 + i] = (float)acc[i];
}

// Symmetric eigen-decomposition (FP64): the published EISPACK method,
// tred2 (Householder reduction to tridiagonal form, accumulating the
// transformations) followed by tql2 (QL iterations with implicit shifts on
// the tridiagonal matrix), in the widely printed tred2/tqli formulation
// (Martin, Reinsch and Wilkinson, Numer. Math. 11 and 12, 1968).  The
// reference's pca.cpp uses Eigen's SelfAdjointEigenSolver, a different
// formulation (tridiagonalisation then implicit symmetric QR steps with a
// Wilkinson shift); both give the eigenpairs to FP64 rounding, which the
// tests check against LAPACK.  Every inner loop walks rows: about 1.3 s at
// d = 960 and a few ms at d = 128.
//
// Householder step: A (d x d, row-major, only its lower triangle used) is
// destroyed; on return A holds Q with A_in = Q T Q^T, diag the diagonal of T
// and off[i] = T[i][i-1] (off[0] = 0).
// Page-aligned, so that neither it nor the QL below crosses a page: with an
// inner loop across a page boundary (wherever the linker happened to put it)
// the fit at d = 960 took 505 ms instead of 378.
constexpr int kCodePage = 4096;
__attribute__((aligned(kCodePage))) static void householder_tridiag(std::vector<double>& A, int d, std::vector<double>& diag,
                                std::vector<double>& off) {
  diag.assign(d, 0.0);
  off.assign(d, 0.0);
  auto a = [&](int i, int j) -> double& { return A[(size_t)i * d + j]; };
  for (int i = d - 1; i > 0; --i) {
    const int l = i - 1;
    double h = 0.0;
    if (l > 0) {
      double scale = 0.0;
      for (int k = 0; k <= l; ++k) scale += fabs(a(i, k));
      if (scale == 0.0) {
        off[i] = a(i, l);
      } else {
        for (int k = 0; k <= l; ++k) {
          a(i, k) /= scale;
          h += a(i, k) * a(i, k);
        }
        const double f = a(i, l);
        const double g = f >= 0.0 ? -sqrt(h) : sqrt(h);
        off[i] = scale * g;
        h -= f * g;
        a(i, l) = f - g;
        // p = A[0..l][0..l] u (u = row i), from the lower triangle row by row
        const double* u = &A[(size_t)i * d];
        for (int j = 0; j <= l; ++j) off[j] = 0.0;
        for (int j = 0; j <= l; ++j) {
          const double* aj = &A[(size_t)j * d];
          double pj = aj[j] * u[j];
          for (int k = 0; k < j; ++k) {
            pj += aj[k] * u[k];
            off[k] += aj[k] * u[j];
          }
          off[j] += pj;
        }
        double ff = 0.0;
        for (int j = 0; j <= l; ++j) {
          a(j, i) = u[j] / h;
          off[j] /= h;
          ff += off[j] * u[j];
        }
        const double hh = ff / (h + h);
        for (int j = 0; j <= l; ++j) {  // A -= u q^T + q u^T on the lower triangle
          const double fj = a(i, j);
          const double gj = off[j] - hh * fj;
          off[j] = gj;
          for (int k = 0; k <= j; ++k) a(j, k) -= fj * off[k] + gj * a(i, k);
        }
      }
    } else {
      off[i] = a(i, l);
    }
    diag[i] = h;
  }
  diag[0] = 0.0;
  off[0] = 0.0;
  // accumulate the reflections into A, which becomes Q
  std::vector<double> gv(d);
  for (int i = 0; i < d; ++i) {
    const int l = i - 1;
    if (diag[i] != 0.0) {
      // g = a(i, 0..l) A[0..l][0..l], then A[k][0..l] -= a(k, i) g, row by row
      for (int j = 0; j <= l; ++j) gv[j] = 0.0;
      for (int k = 0; k <= l; ++k) {
        const double aik = a(i, k);
        const double* ak = &A[(size_t)k * d];
        for (int j = 0; j <= l; ++j) gv[j] += aik * ak[j];
      }
      for (int k = 0; k <= l; ++k) {
        const double aki = a(k, i);
        double* ak = &A[(size_t)k * d];
        for (int j = 0; j <= l; ++j) ak[j] -= aki * gv[j];
      }
    }
    diag[i] = a(i, i);
    a(i, i) = 1.0;
    for (int j = 0; j <= l; ++j) a(j, i) = a(i, j) = 0.0;
  }
}

// QL with implicit shifts on the tridiagonal (diag, off), rotating the rows
// of Zt (row i = vector i, Q^T on entry): on return diag holds the
// eigenvalues and row i of Zt the eigenvector of diag[i].  False if an
// eigenvalue needed more than 60 iterations.
__attribute__((aligned(kCodePage))) static bool tridiag_ql(std::vector<double>& diag, std::vector<double>& off,
                       std::vector<double>& Zt, int d) {
  for (int i = 1; i < d; ++i) off[i - 1] = off[i];
  off[d - 1] = 0.0;
  for (int l = 0; l < d; ++l) {
    int iter = 0;
    int m;
    do {
      for (m = l; m < d - 1; ++m) {  // first negligible off-diagonal element
        const double dd = fabs(diag[m]) + fabs(diag[m + 1]);
        if (fabs(off[m]) <= 1e-15 * dd) break;
      }
      if (m != l) {
        if (iter++ == 60) return false;
        double g = (diag[l + 1] - diag[l]) / (2.0 * off[l]);
        double r = hypot(g, 1.0);
        g = diag[m] - diag[l] + off[l] / (g + (g >= 0.0 ? fabs(r) : -fabs(r)));
        double s = 1.0, c = 1.0, p = 0.0;
        int i;
        for (i = m - 1; i >= l; --i) {
          double f = s * off[i];
          const double b = c * off[i];
          r = hypot(f, g);
          off[i + 1] = r;
          if (r == 0.0) {  // underflow: deflate and restart
            diag[i + 1] -= p;
            off[m] = 0.0;
            break;
          }
          s = f / r;
          c = g / r;
          g = diag[i + 1] - p;
          r = (diag[i] - g) * s + 2.0 * c * b;
          p = s * r;
          diag[i + 1] = g + p;
          g = c * r - b;
          double* zi = &Zt[(size_t)i * d];
          double* zj = zi + d;
          for (int k = 0; k < d; ++k) {
            f = zj[k];
            zj[k] = s * zi[k] + c * f;
            zi[k] = c * zi[k] - s * f;
          }
        }
        if (r == 0.0 && i >= l) continue;
        diag[l] -= p;
        off[l] = g;
        off[m] = 0.0;
      }
    } while (m != l);
  }
  return true;
}

}  // namespace rte

extern "C" {

int rte_pca_fit(rte_ctx* c, const float* X, int64_t n, int d, int64_t stride, float* R_out,
                float* mu_out, double* eig_out, int where) {
  if (!c) return RTE_EINVAL;
  if (!X || !R_out || !mu_out || n < 2 || d < 1 || stride < d)
    return rte_fail(c, RTE_EINVAL, "bad pca arguments");
  if (d > rte::kPcaMaxD) return rte_fail(c, RTE_EUNSUP, "pca for d <= %d (d = %d)", rte::kPcaMaxD, d);
  if (hipSetDevice(c->device) != hipSuccess) return rte_fail(c, RTE_EHIP, "hipSetDevice");
  hipStream_t st = c->stream;
  auto ck = [&](hipError_t e, const char* what) {
    return e == hipSuccess ? RTE_OK : rte_fail(c, RTE_EHIP, "%s: %s", what, hipGetErrorString(e));
  };
  DevBuf xin;
  const float* dx = X;
  if (where == RTE_HOST) {
    const size_t bytes = ((size_t)(n - 1) * stride + d) * sizeof(float);
    if (int r = ck(xin.reserve(bytes), "hipMalloc(pca input)")) return r;
    if (int r = ck(hipMemcpyAsync(xin.p, X, bytes, hipMemcpyHostToDevice, st), "copy")) return r;
    dx = xin.as<float>();
  }
  int cus = 0;
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device);
  cus = std::max(cus, 1);
  const int nt = (d + rte::kPcaTile - 1) / rte::kPcaTile;
  const int ntp = nt * (nt + 1) / 2;
  // row ranges: enough workgroups to fill the chip twice, >= 1024 rows each
  const int64_t by_rows = std::max<int64_t>(1, (n + 1023) / 1024);
  const int nb_sum = (int)std::min<int64_t>(2 * cus, by_rows);
  const int nb = (int)std::min<int64_t>(std::max(1, (2 * cus + ntp - 1) / ntp), by_rows);
  const int64_t rpb_sum = (n + nb_sum - 1) / nb_sum, rpb = (n + nb - 1) / nb;
  const size_t dd = (size_t)d * d;
  // covariance | mean | partials
  const size_t part_n = std::max((size_t)nb * dd, (size_t)nb_sum * d);
  DevBuf work;  // freed on return (hipFree waits for the device)
  if (int r = ck(work.reserve((dd + d + part_n) * sizeof(double)), "hipMalloc(pca work)")) return r;
  double* cov = work.as<double>();
  double* mean = cov + dd;
  double* part = mean + d;
  // whole waves of columns, and no more
  hipLaunchKernelGGL(rte::col_sum_kernel, dim3(nb_sum), dim3(std::min(256, (d + 63) / 64 * 64)), 0,
                     st, dx, n, d, stride,
                     rpb_sum, part);
  hipLaunchKernelGGL(rte::col_mean_kernel, dim3((d + 127) / 128), dim3(128), 0, st,
                     part, nb_sum, d, n, mean);
  hipLaunchKernelGGL(rte::cov_partial_kernel, dim3(nb, ntp), dim3(256), 0, st, dx, n, d, stride,
                     mean, rpb, nt, part);
  hipLaunchKernelGGL(rte::cov_reduce_kernel, dim3((unsigned)((dd + 255) / 256)), dim3(256), 0, st,
                     part, nb, d, n, cov);
  if (int r = ck(hipGetLastError(), "pca kernels")) return r;
  std::vector<double> C(dd), mu(d);
  if (int r = ck(hipMemcpyAsync(C.data(), cov, dd * 8, hipMemcpyDeviceToHost, st), "copy"))
    return r;
  if (int r = ck(hipMemcpyAsync(mu.data(), mean, (size_t)d * 8, hipMemcpyDeviceToHost, st),
                 "copy"))
    return r;
  if (int r = ck(hipStreamSynchronize(st), "sync")) return r;
  std::vector<double> w, off;
  rte::householder_tridiag(C, d, w, off);
  std::vector<double> Zt(dd);  // Q^T: row i = column i of Q
  for (int i = 0; i < d; ++i)
    for (int j = 0; j < d; ++j) Zt[(size_t)j * d + i] = C[(size_t)i * d + j];
  if (!rte::tridiag_ql(w, off, Zt, d))
    return rte_fail(c, RTE_EBUILD, "pca: eigensolver did not converge");
  std::vector<int> order(d);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return w[a] > w[b]; });
  for (int j = 0; j < d; ++j) {
    const double* v = &Zt[(size_t)order[j] * d];
    int arg = 0;  // deterministic sign: largest-magnitude component positive
    for (int i = 1; i < d; ++i)
      if (fabs(v[i]) > fabs(v[arg])) arg = i;
    const double sg = v[arg] < 0 ? -1.0 : 1.0;
    for (int i = 0; i < d; ++i) R_out[(size_t)i * d + j] = (float)(sg * v[i]);
    if (eig_out) eig_out[j] = w[order[j]];
  }
  for (int j = 0; j < d; ++j) mu_out[j] = (float)mu[j];
  return RTE_OK;
}

int rte_pca_rotate(rte_ctx* c, const float* X, int64_t n, int d, int64_t stride, const float* R,
                   const float* mu, int d_out, float* out, int where) {
  if (!c) return RTE_EINVAL;
  if (!X || !R || !mu || !out || n < 0 || d < 1 || d_out < 1 || d_out > d || stride < d)
    return rte_fail(c, RTE_EINVAL, "bad pca_rotate arguments");
  if (n == 0) return RTE_OK;
  if (hipSetDevice(c->device) != hipSuccess) return rte_fail(c, RTE_EHIP, "hipSetDevice");
  hipStream_t st = c->stream;
  auto ck = [&](hipError_t e, const char* what) {
    return e == hipSuccess ? RTE_OK : rte_fail(c, RTE_EHIP, "%s: %s", what, hipGetErrorString(e));
  };
  if ((n + 15) / 16 > 0x7fffffff)
    return rte_fail(c, RTE_EUNSUP, "pca_rotate: too many rows");
  DevBuf xin, rm, ob;
  const float* dx = X;
  float* dout = out;
  const size_t xbytes = ((size_t)(n - 1) * stride + d) * sizeof(float);
  const size_t obytes = (size_t)n * d_out * sizeof(float);
  if (where == RTE_HOST) {
    if (int r = ck(xin.reserve(xbytes), "hipMalloc(pca_rotate input)")) return r;
    if (int r = ck(ob.reserve(obytes), "hipMalloc(pca_rotate output)")) return r;
    if (int r = ck(hipMemcpyAsync(xin.p, X, xbytes, hipMemcpyHostToDevice, st), "copy")) return r;
    dx = xin.as<float>();
    dout = ob.as<float>();
  }
  // R (d x d_out) and mu (d) are host arrays; R widened, where it is, comes first
  // up to 16 columns at any n (1M x 96 to 3: 460 -> 174 us, 20k x 960 to 3: 365 -> 82);
  // up to 32 while there are too few rows to hide the wide kernel's chain (20k x 960
  // to 32: 340 -> 225, 1000 x 128 to 17: 67 -> 50; but 1M x 32 to 32 192 -> 272)
  const bool narrow = d_out <= 16 || (d_out <= 32 && n <= 65536);
  const int ldr = (d_out + rte::kRotCols - 1) / rte::kRotCols * rte::kRotCols;
  const size_t wide = narrow ? 0 : (size_t)(d + 1) * ldr;
  if (int r = ck(rm.reserve(wide * sizeof(double) + ((size_t)d * d_out + d) * sizeof(float)),
                 "hipMalloc"))
    return r;
  double* dW = rm.as<double>();
  float* dR = reinterpret_cast<float*>(dW + wide);
  float* dmu = dR + (size_t)d * d_out;
  if (int r = ck(hipMemcpyAsync(dR, R, (size_t)d * d_out * 4, hipMemcpyHostToDevice, st), "copy"))
    return r;
  if (int r = ck(hipMemcpyAsync(dmu, mu, (size_t)d * 4, hipMemcpyHostToDevice, st), "copy"))
    return r;
  const unsigned blocks = (unsigned)((n + rte::kRotRows - 1) / rte::kRotRows);
  if (narrow) {
    auto* kernel =
        d_out <= 16 ? rte::pca_rotate_narrow_kernel<4> : rte::pca_rotate_narrow_kernel<8>;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, st, dx, n, d, stride, dR, dmu, d_out,
                       dout);
  } else {
    hipLaunchKernelGGL(rte::widen_kernel, dim3((unsigned)((wide + 255) / 256)), dim3(256), 0, st,
                       dR, d, d_out, ldr, dW);
    const int waves = std::min(ldr, rte::kPcaTile) / rte::kRotCols;
    hipLaunchKernelGGL(rte::pca_rotate_kernel,
                       dim3(blocks, (unsigned)((d_out + rte::kPcaTile - 1) / rte::kPcaTile)),
                       dim3(64 * waves), 0, st, dx, n, d, stride, dW, ldr, dmu, d_out, dout);
  }
  if (int r = ck(hipGetLastError(), "pca_rotate kernel")) return r;
  if (where == RTE_HOST) {
    if (int r = ck(hipMemcpyAsync(out, dout, obytes, hipMemcpyDeviceToHost, st), "copy")) return r;
  }
  return ck(hipStreamSynchronize(st), "sync");
}

}  // extern "C"
