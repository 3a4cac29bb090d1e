// Cholesky factor and its inverse of the n x n overlap (rgs), FP64: S = U^T U
// (LAPACK dpotrf, upper) and X = U^-1 (dtrtri), in 64-wide blocks.
//
// The chain of dependent launches bounds it, so each does as much as it can: a
// diagonal block is factored and inverted by one workgroup in LDS, panels of 16 rows
// in the registers of one wave (two barriers per panel), the block row U_kj = X_kk^T
// S_kj uses that inverse, and the launch that updates the trailing blocks also factors
// the next diagonal one.  The off-diagonal blocks of X follow by doubling, X_12 = -X_11
// U_12 X_22.  128 states: 0.13 ms in 6 launches where an LDS element loop with
// three barriers per column, forward substitution per column and one wavefront
// per column of X took 0.31 ms.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mc_internal.h"

namespace mc {

namespace {

constexpr int kCb = 64;          // block edge
constexpr int kLd = kCb + 1;     // LDS row stride

// broadcast of lane `src`'s value (src uniform)
__device__ __forceinline__ double lane_value(double v, int src) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, src), hi = __builtin_amdgcn_readlane((int)(b >> 32), src);
  return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}

// Factors the block T (row-major kCb x kCb with stride kLd in LDS, upper
// triangle used; rows and columns >= nb are those of the identity) into U and
// inverts it: U to S(kb.., kb..) (upper triangle), X to X(kb.., kb..) (whole
// block).  Y: a second LDS block, inv: kCb doubles of LDS.  256 threads.  Panels of 16
// rows: one wave (lane = column) eliminates within the panel in registers, the
// pivot row's entries taken lane by lane, and all waves update the rows behind
// it.  The panel loop stays rolled: fully unrolled, the instructions alone took
// 180 us to fetch (this one: 46, and 12 with one panel).  A pivot that is not positive
// ends the factorisation: *info = its order.
__device__ void factor_block(double* T, double* Y, double* inv, int nb, int kb, double* __restrict__ S, int lds,
                             double* __restrict__ X, int ldx, int* info, int* bad) {
  constexpr int kP = 16;
  const int w = threadIdx.x >> 6, c = threadIdx.x & 63;
  const int np = (nb + kP - 1) / kP * kP;   // the panels behind are those of the identity
  if (threadIdx.x == 0) *bad = 0;
  for (int e = threadIdx.x; e < kCb * kCb; e += 256) {
    const int r = e / kCb, cc = e & (kCb - 1);
    Y[r * kLd + cc] = r == cc ? 1.0 : 0.0;
  }
  __syncthreads();
#pragma unroll 1
  for (int r0 = 0; r0 < np; r0 += kP) {
    if (w == 0) {
      double t[kP];
#pragma unroll
      for (int i = 0; i < kP; ++i) t[i] = T[(r0 + i) * kLd + c];
#pragma unroll
      for (int j = 0; j < kP; ++j) {
        const double d = lane_value(t[j], r0 + j);
        if (!(d > 0.0) && c == 0 && *bad == 0) *bad = kb + r0 + j + 1;
        const double rs = rsqrt(d);
        if (c == 0) inv[r0 + j] = rs;
        t[j] *= rs;
#pragma unroll
        for (int r = j + 1; r < kP; ++r) t[r] -= lane_value(t[j], r0 + r) * t[j];
      }
#pragma unroll
      for (int i = 0; i < kP; ++i) T[(r0 + i) * kLd + c] = c >= r0 + i ? t[i] : 0.0;
    }
    __syncthreads();
    double u[kP];
#pragma unroll
    for (int j = 0; j < kP; ++j) u[j] = T[(r0 + j) * kLd + c];
#pragma unroll 1
    for (int r = r0 + kP + w; r < np; r += 4) {
      double a = T[r * kLd + c];
#pragma unroll
      for (int j = 0; j < kP; ++j) a -= T[(r0 + j) * kLd + r] * u[j];
      T[r * kLd + c] = a;
    }
    __syncthreads();
  }
  if (*bad) {   // uniform
    if (threadIdx.x == 0) *info = *bad;
    return;
  }
  for (int e = threadIdx.x; e < kCb * kCb; e += 256) {
    const int r = e & (kCb - 1), cc = e / kCb;
    if (r <= cc && cc < nb) S[(size_t)lds * (kb + cc) + kb + r] = T[r * kLd + cc];
  }
  // X = U^-1 by columns, panels from the last: x_k = b_k / U_kk, b_r -= U_rk x_k
#pragma unroll 1
  for (int r0 = np - kP; r0 >= 0; r0 -= kP) {
    if (w == 0) {
      double t[kP], b[kP];
#pragma unroll
      for (int i = 0; i < kP; ++i) {
        t[i] = T[(r0 + i) * kLd + c];
        b[i] = Y[(r0 + i) * kLd + c];
      }
#pragma unroll
      for (int k = kP - 1; k >= 0; --k) {
        b[k] *= inv[r0 + k];
#pragma unroll
        for (int r = 0; r < k; ++r) b[r] -= lane_value(t[r], r0 + k) * b[k];
      }
#pragma unroll
      for (int i = 0; i < kP; ++i) Y[(r0 + i) * kLd + c] = b[i];
    }
    __syncthreads();
    double x[kP];
#pragma unroll
    for (int k = 0; k < kP; ++k) x[k] = Y[(r0 + k) * kLd + c];
#pragma unroll 1
    for (int r = w; r < r0; r += 4) {
      double a = Y[r * kLd + c];
#pragma unroll
      for (int k = 0; k < kP; ++k) a -= T[r * kLd + r0 + k] * x[k];
      Y[r * kLd + c] = a;
    }
    __syncthreads();
  }
  for (int e = threadIdx.x; e < kCb * kCb; e += 256) {
    const int r = e & (kCb - 1), cc = e / kCb;
    if (r < nb && cc < nb) X[(size_t)ldx * (kb + cc) + kb + r] = r <= cc ? Y[r * kLd + cc] : 0.0;
  }
}

// nr x nc block of a column-major matrix into LDS, T[r][c], zero beyond it; all
// 16 loads of a thread in flight (indices beyond the block repeat its last ones)
__device__ __forceinline__ void load_block(double* T, const double* __restrict__ M, int ld, int nr, int nc) {
  double v[16];
  const int r = threadIdx.x & (kCb - 1), c0 = threadIdx.x / kCb;
#pragma unroll
  for (int u = 0; u < 16; ++u) v[u] = M[(size_t)ld * min(c0 + 4 * u, nc - 1) + min(r, nr - 1)];
#pragma unroll
  for (int u = 0; u < 16; ++u) T[r * kLd + c0 + 4 * u] = r < nr && c0 + 4 * u < nc ? v[u] : 0.0;
}

// thread (ty, tx) of 16 x 16 holds the results (ty + 16 a, tx + 16 b):
// acc += sum_k A(k, i) B(k, j) with both blocks as [k][.]
__device__ __forceinline__ void mult_tn(const double* A, const double* B, double (&acc)[4][4]) {
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
#pragma unroll 4
  for (int k = 0; k < kCb; ++k) {
    double a[4], b[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      a[u] = A[k * kLd + ty + 16 * u];
      b[u] = B[k * kLd + tx + 16 * u];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[u][v] += a[u] * b[v];
  }
}
// acc += sum_k A(i, k) B(k, j), A as [i][k]
__device__ __forceinline__ void mult_nn(const double* A, const double* B, double (&acc)[4][4]) {
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
#pragma unroll 4
  for (int k = 0; k < kCb; ++k) {
    double a[4], b[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      a[u] = A[(ty + 16 * u) * kLd + k];
      b[u] = B[k * kLd + tx + 16 * u];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[u][v] += a[u] * b[v];
  }
}

// first diagonal block; clears *info
__global__ __launch_bounds__(256) void k_chol_first(double* __restrict__ S, int lds, int n, double* __restrict__ X,
                                                    int ldx, int* info) {
  __shared__ double T[kCb * kLd];
  __shared__ double Y[kCb * kLd];
  __shared__ double inv[kCb];
  __shared__ int bad;
  const int nb = min(kCb, n);
  load_block(T, S, lds, nb, nb);   // the lower triangle is not used
  __syncthreads();
  if (threadIdx.x >= nb && threadIdx.x < kCb) T[threadIdx.x * kLd + threadIdx.x] = 1.0;
  if (threadIdx.x == 0) *info = 0;
  __syncthreads();
  factor_block(T, Y, inv, nb, 0, S, lds, X, ldx, info, &bad);
}

// block row k: U_kj = X_kk^T S_kj for the 64-column blocks j > k (one each)
__global__ __launch_bounds__(256) void k_chol_row(double* __restrict__ S, int lds, int n, int kb,
                                                  const double* __restrict__ X, int ldx, const int* info) {
  __shared__ double A[kCb * kLd];
  __shared__ double B[kCb * kLd];
  if (*info) return;
  const int j0 = kb + kCb * (1 + blockIdx.x), nc = min(kCb, n - j0);
  double* Sj = S + (size_t)lds * j0 + kb;
  load_block(A, X + (size_t)ldx * kb + kb, ldx, kCb, kCb);
  load_block(B, Sj, lds, kCb, nc);
  __syncthreads();
  double acc[4][4] = {};
  mult_tn(A, B, acc);
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
#pragma unroll
  for (int v = 0; v < 4; ++v)
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (tx + 16 * v < nc) Sj[(size_t)lds * (tx + 16 * v) + ty + 16 * u] = acc[u][v];
}

// trailing update S_ij -= U_ki^T U_kj, blocks k < i <= j, linear over the upper
// triangle; the workgroup of block (k+1, k+1) factors it
__global__ __launch_bounds__(256) void k_chol_update(double* __restrict__ S, int lds, int n, int kb,
                                                     double* __restrict__ X, int ldx, int* info) {
  __shared__ double A[kCb * kLd];
  __shared__ double B[kCb * kLd];
  __shared__ double inv[kCb];
  __shared__ int bad;
  // only the workgroup that may set *info looks at it: for the others it could change
  // between two of their waves (what they form after a failure is not used)
  if (blockIdx.x == 0 && *info) return;
  const int nt = (n - kb - 1) / kCb;   // block columns behind k
  int ti, tj;
  tile_ij(blockIdx.x, true, nt, nt, ti, tj);
  const int i0 = kb + kCb * (1 + ti), j0 = kb + kCb * (1 + tj);
  const int nr = min(kCb, n - i0), nc = min(kCb, n - j0);
  load_block(A, S + (size_t)lds * i0 + kb, lds, kCb, nr);
  load_block(B, S + (size_t)lds * j0 + kb, lds, kCb, nc);
  __syncthreads();
  double acc[4][4] = {};
  mult_tn(A, B, acc);
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  double* Sij = S + (size_t)lds * j0 + i0;
  const bool next = blockIdx.x == 0;   // tile (0, 0)
  if (next) __syncthreads();           // A becomes the block to factor
#pragma unroll
  for (int v = 0; v < 4; ++v)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = ty + 16 * u, c = tx + 16 * v;
      const bool in = r < nr && c < nc;
      if (next) {
        A[r * kLd + c] = in ? (r <= c ? Sij[(size_t)lds * c + r] - acc[u][v] : 0.0) : (r == c ? 1.0 : 0.0);
      } else if (in) {
        Sij[(size_t)lds * c + r] -= acc[u][v];
      }
    }
  if (next) {
    __syncthreads();
    factor_block(A, B, inv, nr, i0, S, lds, X, ldx, info, &bad);
  }
}

// One doubling step of X = U^-1 from blocks of s rows to 2 s: pair p covers the
// rows o = 2 s p .. (first part s, second n2 <= s).  STEP 0: W_12 = U_12 X_22,
// at the place of U_12; STEP 1: X_12 = -X_11 W_12.  Workgroup (64
// x 64 tile, pair); the triangular factor's zero blocks are skipped.
template <int STEP>
__global__ __launch_bounds__(256) void k_tri_double(const double* __restrict__ U, int ldu, int n, int s,
                                                    double* __restrict__ X, int ldx, double* __restrict__ W, int ldw,
                                                    const int* info) {
  __shared__ double A[kCb * kLd];
  __shared__ double B[kCb * kLd];
  if (*info) return;
  const int o = 2 * s * blockIdx.z, m0 = o + s;
  const int n2 = min(s, n - m0);
  const int r0 = kCb * blockIdx.x, c0 = kCb * blockIdx.y;   // tile within the s x n2 block
  if (n2 <= 0 || c0 >= n2) return;
  const int nc = min(kCb, n2 - c0);
  double acc[4][4] = {};
  // STEP 0: k over the rows of X_22 up to the tile's columns; STEP 1: over the
  // columns of X_11 from the tile's rows
  const int k0 = STEP == 0 ? 0 : r0, k1 = STEP == 0 ? min(n2, c0 + kCb) : s;
  for (int k = k0; k < k1; k += kCb) {
    const int nk = min(kCb, k1 - k);
    if (k > k0) __syncthreads();
    if constexpr (STEP == 0) {
      load_block(A, U + (size_t)ldu * (m0 + k) + o + r0, ldu, kCb, nk);
      load_block(B, X + (size_t)ldx * (m0 + c0) + m0 + k, ldx, nk, nc);
    } else {
      load_block(A, X + (size_t)ldx * (o + k) + o + r0, ldx, kCb, nk);
      load_block(B, W + (size_t)ldw * (m0 + c0) + o + k, ldw, nk, nc);
    }
    __syncthreads();
    mult_nn(A, B, acc);
  }
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  double* out = STEP == 0 ? W + (size_t)ldw * (m0 + c0) + o + r0 : X + (size_t)ldx * (m0 + c0) + o + r0;
  const int ld = STEP == 0 ? ldw : ldx;
#pragma unroll
  for (int v = 0; v < 4; ++v)
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (tx + 16 * v < nc) out[(size_t)ld * (tx + 16 * v) + ty + 16 * u] = STEP == 0 ? acc[u][v] : -acc[u][v];
}

}  // namespace

void chol_inverse(mc_ctx* ctx, double* S, int n, double* X, double* W, int* info) {
  hipLaunchKernelGGL(k_zero, dim3(256), dim3(256), 0, ctx->stream, X, (size_t)n * n);
  MC_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_chol_first, dim3(1), dim3(256), 0, ctx->stream, S, n, n, X, n, info);
  MC_HIP(hipGetLastError());
  for (int kb = 0; kb + kCb < n; kb += kCb) {
    const int nt = (n - kb - 1) / kCb;
    hipLaunchKernelGGL(k_chol_row, dim3(nt), dim3(256), 0, ctx->stream, S, n, n, kb, X, n, info);
    MC_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_chol_update, dim3(nt * (nt + 1) / 2), dim3(256), 0, ctx->stream, S, n, n, kb, X, n, info);
    MC_HIP(hipGetLastError());
  }
  for (int s = kCb; s < n; s *= 2) {
    const dim3 g(s / kCb, s / kCb, (n - s + 2 * s - 1) / (2 * s));
    hipLaunchKernelGGL(k_tri_double<0>, g, dim3(256), 0, ctx->stream, S, n, n, s, X, n, W, n, info);
    MC_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_tri_double<1>, g, dim3(256), 0, ctx->stream, S, n, n, s, X, n, W, n, info);
    MC_HIP(hipGetLastError());
  }
}

}  // namespace mc
