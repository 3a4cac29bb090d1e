// S^-1/2 of an overlap matrix by the coupled Newton-Schulz iteration, FP64
// (lowdin, src/lowdin_utils.mod.F90):
//
//   Y_0 = S/c, Z_0 = I;  T = 3/2 I - 1/2 Z Y,  Y <- Y T,  Z <- T Z;  Z -> sqrt(c) S^-1/2
//
// The iterates commute and are symmetric only up to rounding, and the iteration is
// stable only while its products are those of the factors as they are, in this order:
// formed as A^T B, or from the tiles above the diagonal mirrored below it, they
// amplify the commutator, and S of a condition of 1e2 or 1e3 diverges (with true
// products it converges to 1e6 and beyond).  So every tile is formed, A read by its rows.
//
// At a few hundred states a product is bound by latency, not by the matrix cores
// (512: 0.27 GF, 4 us at 68 TF/s): it has to be cut into enough workgroups.  k_product
// takes 32 x 32 tiles (256 at 512), the K range split over the four waves of a
// workgroup and added in LDS, operands straight from L2 into registers one group of 32
// k ahead.  Its epilogue forms T and the largest |T - I|, and the products Y T and T Z
// share a launch, so that an iteration is two launches (as three general products of 36
// us with 64 workgroups, two copies, two element passes, a reduction and a wait of the
// host it took 160 us at 512 states).  lowdin of 67 states: 0.53 -> 0.17 ms; 512 / 1024 /
// 4096 states over 12,443 / 17,133 plane waves 2.2 / 6.6 / 151 -> 0.9 / 3.7 / 114 ms.  The
// host reads max |T - I| while the next iteration runs, which is needed in any case: one
// more follows the one that has converged.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "mc_internal.h"

namespace mc {

namespace {

typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kPad = 128;   // K rows are padded (with zeros) to four waves of 32

// colsum[j] = sum_i |S(i, j)|, colsum[n + j] = sum_i S(i, j)^2; one workgroup per column
__global__ __launch_bounds__(256) void k_col_norms(const double* __restrict__ S, int n, double* __restrict__ colsum) {
  const int j = blockIdx.x;
  double a = 0.0, q = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) {
    const double v = S[i + (size_t)j * n];
    a += fabs(v);
    q += v * v;
  }
  __shared__ double sa[256], sq[256];
  sa[threadIdx.x] = a;
  sq[threadIdx.x] = q;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) {
      sa[threadIdx.x] += sa[threadIdx.x + h];
      sq[threadIdx.x] += sq[threadIdx.x + h];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    colsum[j] = sa[0];
    colsum[n + j] = sq[0];
  }
}

// Y0 = s S, Z0 = I with zeros behind row and column n; Y1, Z1, T zero; dev slots zero
__global__ void k_start(const double* __restrict__ S, int n, int ld, double s, double* __restrict__ Y0,
                        double* __restrict__ Z0, double* __restrict__ rest, unsigned long long* __restrict__ dev,
                        int ndev) {
  const size_t nn = (size_t)ld * ld;
  for (size_t e = blockIdx.x * 256 + threadIdx.x; e < nn; e += (size_t)gridDim.x * 256) {
    const int j = (int)(e / ld), i = (int)(e - (size_t)j * ld);
    const bool in = i < n && j < n;
    Y0[e] = in ? s * S[i + (size_t)j * n] : 0.0;
    Z0[e] = in && i == j ? 1.0 : 0.0;
    for (int r = 0; r < 3; ++r) rest[r * nn + e] = 0.0;
    if (e < (size_t)ndev) dev[e] = 0;
  }
}

__global__ void k_finish(const double* __restrict__ Z, int n, int ld, double s, double* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x, j = blockIdx.y;
  if (i < n) out[i + (size_t)j * n] = s * Z[i + (size_t)j * ld];
}

struct Product {
  const double* a;
  const double* b;
  double* d;
};

// d = alpha a b + beta I (n x n, ld a multiple of kPad, zero behind n); blockIdx.x =
// tile, blockIdx.y = product.  dev (may be null): the bits of max |d - I|, which order
// like the values, with NaN above all.
__global__ __launch_bounds__(256) void k_product(Product p0, Product p1, int n, int ld, int nt, double alpha,
                                                 double beta, unsigned long long* __restrict__ dev) {
  __shared__ double part[4][32 * 33];
  const Product p = blockIdx.y ? p1 : p0;
  const int i0 = 32 * ((int)blockIdx.x % nt), j0 = 32 * ((int)blockIdx.x / nt);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
  const int per = ld / 4, k0 = wave * per;
  // a by rows: a lane holds the rows 2 li, 2 li + 1 of one k (a column's 32 rows are 256
  // contiguous bytes); b by columns j0 + li, + 16, two k at a time
  const double* pa = p.a + i0 + 2 * li + (size_t)(k0 + 2 * lq) * ld;
  const double* pb = p.b + (size_t)(j0 + li) * ld + k0 + 2 * lq;
  const size_t c16 = (size_t)16 * ld;
  d2 f[2][4][4];   // [stage][step of 8 k][a at k = 2 lq, 2 lq + 1, b0, b1]
  const auto load = [&](int k, int st) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      f[st][u][0] = *reinterpret_cast<const d2*>(pa + (size_t)(k + 8 * u) * ld);
      f[st][u][1] = *reinterpret_cast<const d2*>(pa + (size_t)(k + 8 * u + 1) * ld);
      f[st][u][2] = *reinterpret_cast<const d2*>(pb + k + 8 * u);
      f[st][u][3] = *reinterpret_cast<const d2*>(pb + c16 + k + 8 * u);
    }
  };
  d4 acc[2][2];   // [row of the pair][column block]
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = d4{0.0, 0.0, 0.0, 0.0};
  const auto multiply = [&](int st) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b)
            acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(a ? f[st][u][s].y : f[st][u][s].x,
                                                             s ? f[st][u][2 + b].y : f[st][u][2 + b].x, acc[a][b], 0, 0, 0);
  };
  load(0, 0);
  int k = 0;
  for (; k + 64 <= per; k += 64) {   // two groups of 32 k
    load(k + 32, 1);
    multiply(0);
    if (k + 64 < per) load(k + 64, 0);
    multiply(1);
  }
  if (k < per) multiply(0);
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[wave][(16 * b + li) * 33 + 2 * (4 * r + lq) + a] = acc[a][b][r];
  __syncthreads();
  double big = 0.0;
  bool bad = false;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int x = threadIdx.x & 31, y = (threadIdx.x >> 5) + 8 * q, e = y * 33 + x;
    if (i0 + x >= n || j0 + y >= n) continue;
    const double one = i0 + x == j0 + y ? 1.0 : 0.0;
    const double v = alpha * ((part[0][e] + part[1][e]) + (part[2][e] + part[3][e])) + one * beta;
    p.d[i0 + x + (size_t)(j0 + y) * ld] = v;
    const double t = fabs(v - one);
    bad |= t != t;
    big = fmax(big, t);
  }
  if (!dev) return;
  if (bad) big = __longlong_as_double(0x7ff8000000000000LL);
  unsigned long long m = (unsigned long long)__double_as_longlong(big);
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long w = __shfl_xor(m, o);
    m = w > m ? w : m;
  }
  if (lane == 0) atomicMax(dev, m);
}

// *src once the stream has reached this point; more() is enqueued behind the copy
// before the host waits
template <typename F>
double read_behind(mc_ctx* ctx, const double* src, F&& more) {
  double* h = static_cast<double*>(ctx->h_down);   // allocated by the dl_add above, nothing pending
  if (!ctx->h_down_done) MC_HIP(hipEventCreateWithFlags(&ctx->h_down_done, hipEventDisableTiming));
  MC_HIP(hipMemcpyAsync(h, src, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  MC_HIP(hipEventRecord(ctx->h_down_done, ctx->stream));
  more();
  MC_HIP(hipEventSynchronize(ctx->h_down_done));
  return *h;
}

}  // namespace

void inv_sqrt(mc_ctx* ctx, const double* S, int n, double* Zout, int* iters) {
  constexpr int maxit = 100;
  const int ld = (n + kPad - 1) / kPad * kPad, nt = (n + 31) / 32;
  const size_t nn = (size_t)ld * ld;
  // Y, Z (two each), T, column norms, max |T - I| of each iteration, where the
  // overlap's partials were (S holds their sum)
  ctx->w_gemm.ensure(sizeof(double) * (5 * nn + 2 * (size_t)n + maxit + 1));
  double* Y[2] = {ctx->w_gemm.as<double>(), ctx->w_gemm.as<double>() + 2 * nn};
  double* Z[2] = {Y[0] + nn, Y[0] + 3 * nn};
  double* T = Y[0] + 4 * nn;
  double* col = T + nn;
  unsigned long long* dev = reinterpret_cast<unsigned long long*>(col + 2 * (size_t)n);
  hipLaunchKernelGGL(k_col_norms, dim3(n), dim3(256), 0, ctx->stream, S, n, col);
  MC_HIP(hipGetLastError());
  std::vector<double> h(2 * (size_t)n);
  dl_add(ctx, h.data(), col, sizeof(double) * h.size());
  dl_finish(ctx);
  double fro = 0.0, cmax = 0.0;
  for (int j = 0; j < n; ++j) {
    fro += h[n + j];
    cmax = std::max(cmax, h[j]);
  }
  fro = std::sqrt(fro);
  MC_CHECK(fro > 0.0 && std::isfinite(fro), MC_ERR_ARG, "lowdin: zero or non-finite overlap matrix");
  const double c = cmax > 1.0 ? cmax : 1.0;   // ||S||_2 <= ||S||_1 (symmetric): ||I - S/c||_2 < 1
  hipLaunchKernelGGL(k_start, dim3((unsigned)std::min<size_t>(1024, (nn + 255) / 256)), dim3(256), 0, ctx->stream, S, n,
                     ld, 1.0 / c, Y[0], Z[0], Y[1], dev, maxit + 1);
  MC_HIP(hipGetLastError());
  const auto sweep = [&](int it) {   // iterate it from the buffers (it - 1) % 2
    const int o = (it - 1) & 1, w = it & 1;
    const Product zy = {Z[o], Y[o], T}, yt = {Y[o], T, Y[w]}, tz = {T, Z[o], Z[w]};
    hipLaunchKernelGGL(k_product, dim3(nt * nt), dim3(256), 0, ctx->stream, zy, zy, n, ld, nt, -0.5, 1.5, dev + it);
    hipLaunchKernelGGL(k_product, dim3(nt * nt, 2), dim3(256), 0, ctx->stream, yt, tz, n, ld, nt, 1.0, 0.0,
                       (unsigned long long*)nullptr);
    MC_HIP(hipGetLastError());
  };
  sweep(1);
  bool done = false;
  int it = 1;
  for (; it <= maxit; ++it) {
    const double d = read_behind(ctx, reinterpret_cast<const double*>(dev + it), [&] {
      if (it < maxit) sweep(it + 1);
    });
    MC_CHECK(std::isfinite(d), MC_ERR_NOCONV, "lowdin: Newton-Schulz iteration diverged");
    if (d < 1e-15 * n) {   // the correction is at rounding level: the sweep behind it is the last
      done = true;
      ++it;
      break;
    }
  }
  MC_CHECK(done, MC_ERR_NOCONV, "lowdin: Newton-Schulz iteration did not converge in 100 steps");
  hipLaunchKernelGGL(k_finish, dim3((n + 255) / 256, n), dim3(256), 0, ctx->stream, Z[std::min(it, maxit) & 1], n, ld,
                     1.0 / std::sqrt(c), Zout);
  MC_HIP(hipGetLastError());
  if (iters) *iters = it;
}

}  // namespace mc
