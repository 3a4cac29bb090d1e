// FP64 MFMA contractions of 16-byte aligned operands (v_mfma_f64_16x16x4_f64):
// the wavefunction products of the FP64 path.
//
//   k_tn_f64: partials of A^T B over K (both operands K-contiguous columns),
//             A optionally the nonlocal projectors built on the fly;
//   k_nn_f64: D = alpha A G + beta D with A (M x k) tall, G (k x n) small,
//             A optionally the projectors (fnonloc).
//
// A workgroup of 4 waves (2 x 2) computes 32 NI x 32 NJ of the result, a wave
// 16 NI x 16 NJ of it; the tile edges follow the result's (tile_width,
// nn_width).  K advances in
// slices of 16 through two LDS stages.  Both operands of a slice are copied
// straight to LDS 16 bytes per lane (global_load_lds_dwordx4), in 1 KiB runs
// that cover whole 128-byte lines, while the slice before is multiplied.  Both
// are bound by the matrix cores: at 512 states and 396,408 rows a full A^T B
// takes 3.11 ms (67 TF/s; a 512 x 512 x 396408 library product reaches 58, the
// instruction alone 68) and the symmetric one 2.01 ms, A G with its n x n factor
// 3.41 ms (61 TF/s).  The kernels before (8-byte strided loads through
// registers, 64 lines touched per load instruction: bound by the address unit)
// took 5.37, 3.52 and 4.51 ms.
// LDS is read through vector types and the slice cut by the end of K is staged
// apart from the loop: otherwise the compiler waits for all outstanding copies
// before the first read of every slice.
//
// Contraction order: the k pairs of a 16-byte chunk go to consecutive MFMAs
// (lane group q holds k = 8h + 2q + s in step (h, s)), for A and B alike; A G
// stages G so that they are k = 8h + 4s + q.
//
// MFMA operand layout (16x16x4 f64, checked on gfx950 with a lane probe):
// lane l holds A[i = l%16][k = l/16], B[k = l/16][j = l%16] and, in
// accumulator register r, D[i = 4r + l/16][j = l%16].  The small operand (B of
// A^T B, G) is passed first, so that the 16 lanes of a register run along the
// columns' contiguous index and results are stored without an LDS stage.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mc_internal.h"

namespace mc {

namespace {

typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kKs = 16;       // K slice: 128 bytes of a column, 8 chunks of 16 bytes
constexpr int kXcds = 8;

// 16 bytes per lane from src straight into LDS at dst + 16 * lane (dst uniform
// over the wave)
__device__ __forceinline__ void copy16_lds(const void* src, lds_void* dst) {
  __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
}

// this wave's copies have landed and its LDS reads are done, then all waves'
// (s_waitcnt vmcnt(0) lgkmcnt(0), gfx9 encoding)
__device__ __forceinline__ void slice_barrier() {
  __builtin_amdgcn_s_waitcnt(0x70);
  asm volatile("s_barrier" ::: "memory");
}

// chunk q (k = 2q, 2q + 1 of the slice) of column c sits at 16-byte slot
// 8c + (q ^ (c/2 mod 8)): 16 consecutive columns at one q fall on 16 distinct
// slots of the 256-byte bank row
__device__ __forceinline__ int chunk_slot(int c, int q) { return 8 * c + (q ^ ((c >> 1) & 7)); }

// workgroup id -> tile: XCD x = id % 8 gets the contiguous range [x per, (x+1) per)
__device__ __forceinline__ int xcd_index(int total) {
  const int per = (total + kXcds - 1) / kXcds;
  return (int)(blockIdx.x % kXcds) * per + (int)(blockIdx.x / kXcds);
}

// Projector column `col`: (-i)^l twnl(g) [gk(g)] eigr(g), G = 0 halved if
// g0half.  Raw holds the loads of one G vector, so that they can be in flight
// while the slice before is multiplied.
struct ProjCol {
  const d2* e;
  const double* tw;
  const double* gk;   // twnl again where the column has no gk factor (not used then)
  int l;              // l mod 4 of (-i)^l; bit 2: times gk
};
struct Raw {
  d2 e;
  double tw, gk;
};
__device__ __forceinline__ ProjCol proj_col(const ProjTab& t, int col) {
  const int v = t.v0 + col / t.ncol;   // 0: fnl, 1..3: dfnl along x, y, z
  const int4 d = t.tab[col % t.ncol];
  ProjCol p;
  p.e = reinterpret_cast<const d2*>(t.eigr) + (size_t)d.x * t.ldg;
  p.tw = t.twnl + (size_t)d.y * t.ldg;
  p.gk = v > 0 ? t.gk + (size_t)(v - 1) * t.ldg : p.tw;
  p.l = ((d.z + (v > 0 ? 1 : 0)) & 3) | (v > 0 ? 4 : 0);
  return p;
}
__device__ __forceinline__ Raw proj_load(const ProjCol& p, int g) { return Raw{p.e[g], p.tw[g], p.gk[g]}; }
__device__ __forceinline__ d2 proj_value(const Raw& r, int l, bool half) {
  double tw = (l & 4) ? r.tw * r.gk : r.tw;
  if (half) tw *= 0.5;
  if (l & 2) tw = -tw;
  return (l & 1) ? d2{tw * r.e.y, -tw * r.e.x} : d2{tw * r.e.x, tw * r.e.y};
}

// ---------------------------------------------------------------------------
// A^T B partials: P[s] (m x n column-major) over K rows [s kchunk, (s+1) kchunk).
// Launch ceil(total/8)*8 workgroups, total = nsplit * tiles; upper (m == n,
// NI == NJ): only the tiles on or above the diagonal.
// ---------------------------------------------------------------------------
template <int NI, int NJ, bool PROJ>
__global__ __launch_bounds__(256, 2) void k_tn_f64(const double* __restrict__ A, int lda,
                                                   const double* __restrict__ B, int ldb, int K, int m, int n,
                                                   int kchunk, double* __restrict__ P, int upper, ProjTab proj,
                                                   int tm, int tn, int total) {
  constexpr int TI = 32 * NI, TJ = 32 * NJ;   // tile of the result
  constexpr int kStage = (TI + TJ) * 128;     // bytes of one stage
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * kStage];
  const int t = xcd_index(total);
  if (t >= total) return;
  const int tiles = tile_count(upper, tm, tn);
  const int sp = t / tiles;
  int ti, tj;
  tile_ij(t - sp * tiles, upper, tm, tn, ti, tj);
  const int i0 = ti * TI, j0 = tj * TJ;
  const int kbeg = sp * kchunk, kend = min(K, kbeg + kchunk);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // copies: run r of an operand (1 KiB) holds its columns 8r .. 8r+7; wave w
  // copies the runs w, w + 4, ...; lane -> column lane/8 and the chunk that
  // belongs in slot lane%8.  Columns beyond m or n repeat the last one: their
  // results are not stored.
  const int cl = lane >> 3;
  const int q = (lane & 7) ^ ((4 * (wave & 1) + (cl >> 1)) & 7);
  const double* pa[NI];
  const double* pb[NJ];
  ProjCol pc[NI];
#pragma unroll
  for (int u = 0; u < NI; ++u) {
    const int col = min(i0 + 8 * (wave + 4 * u) + cl, m - 1);
    if constexpr (PROJ) pc[u] = proj_col(proj, col);
    else pa[u] = A + (size_t)col * lda + 2 * q;
  }
#pragma unroll
  for (int u = 0; u < NJ; ++u) pb[u] = B + (size_t)min(j0 + 8 * (wave + 4 * u) + cl, n - 1) * ldb + 2 * q;
  Raw ra[NI];
  int ga = 0;   // G vector of ra
  // copies of the whole slice at kb into stage st (a projector operand is
  // fetched into registers and put there by put_a)
  auto issue = [&](int kb, int st) {
    unsigned char* sa = lds + st * kStage;
    unsigned char* sb = sa + TI * 128;
    if constexpr (PROJ) ga = (kb >> 1) + q;
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      if constexpr (PROJ) ra[u] = proj_load(pc[u], ga);
      else copy16_lds(pa[u] + kb, (lds_void*)(sa + (wave + 4 * u) * 1024));
    }
#pragma unroll
    for (int u = 0; u < NJ; ++u) copy16_lds(pb[u] + kb, (lds_void*)(sb + (wave + 4 * u) * 1024));
  };
  auto put_a = [&](int st) {
    if constexpr (PROJ) {
      unsigned char* sa = lds + st * kStage;
#pragma unroll
      for (int u = 0; u < NI; ++u)
        *reinterpret_cast<d2*>(sa + (wave + 4 * u) * 1024 + lane * 16) =
            proj_value(ra[u], pc[u].l, proj.geq0 && ga == 0);
    }
  };
  const int wr = (wave >> 1) * 16 * NI, wc = (wave & 1) * 16 * NJ;
  const int li = lane & 15, lq = lane >> 4;
  d4 acc[NI][NJ];
#pragma unroll
  for (int a = 0; a < NI; ++a)
#pragma unroll
    for (int b = 0; b < NJ; ++b) acc[a][b] = d4{0.0, 0.0, 0.0, 0.0};
  auto multiply = [&](int st) {
    const unsigned char* sa = lds + st * kStage;
    const unsigned char* sb = sa + TI * 128;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      d2 fa[NI], fb[NJ];
#pragma unroll
      for (int a = 0; a < NI; ++a)
        fa[a] = *reinterpret_cast<const d2*>(sa + 16 * chunk_slot(wr + 16 * a + li, 4 * h + lq));
#pragma unroll
      for (int b = 0; b < NJ; ++b)
        fb[b] = *reinterpret_cast<const d2*>(sb + 16 * chunk_slot(wc + 16 * b + li, 4 * h + lq));
#pragma unroll
      for (int b = 0; b < NJ; ++b)
#pragma unroll
        for (int a = 0; a < NI; ++a)
          acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[b].x, fa[a].x, acc[a][b], 0, 0, 0);
#pragma unroll
      for (int b = 0; b < NJ; ++b)
#pragma unroll
        for (int a = 0; a < NI; ++a)
          acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[b].y, fa[a].y, acc[a][b], 0, 0, 0);
    }
  };
  const int nfull = (kend - kbeg) / kKs;   // kbeg < kend for every workgroup
  if (nfull > 0) {
    issue(kbeg, 0);
    put_a(0);
  }
  int st = 0;
  for (int i = 0; i < nfull; ++i, st ^= 1) {
    slice_barrier();   // slice i is staged, and every wave is done with the other stage
    const bool more = i + 1 < nfull;
    if (more) issue(kbeg + (i + 1) * kKs, st ^ 1);
    multiply(st);
    if (more) put_a(st ^ 1);
  }
  if (kbeg + nfull * kKs < kend) {   // the slice cut by kend: rows beyond it count as zero
    const int kb = kbeg + nfull * kKs, k = kb + 2 * q;
    unsigned char* sa = lds + st * kStage;
    unsigned char* sb = sa + TI * 128;
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      d2 v = {0.0, 0.0};
      if constexpr (PROJ) {
        if (k < kend) v = proj_value(proj_load(pc[u], k >> 1), pc[u].l, proj.geq0 && k == 0);
      } else {
        if (k < kend) v.x = pa[u][kb];
        if (k + 1 < kend) v.y = pa[u][kb + 1];
      }
      *reinterpret_cast<d2*>(sa + (wave + 4 * u) * 1024 + lane * 16) = v;
    }
#pragma unroll
    for (int u = 0; u < NJ; ++u) {
      d2 v = {0.0, 0.0};
      if (k < kend) v.x = pb[u][kb];
      if (k + 1 < kend) v.y = pb[u][kb + 1];
      *reinterpret_cast<d2*>(sb + (wave + 4 * u) * 1024 + lane * 16) = v;
    }
    __syncthreads();
    multiply(st);
  }
  double* Ps = P + (size_t)sp * m * n;
#pragma unroll
  for (int a = 0; a < NI; ++a) {
    const int i = i0 + wr + 16 * a + li;
#pragma unroll
    for (int b = 0; b < NJ; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = j0 + wc + 16 * b + 4 * r + lq;
        if (i < m && j < n) Ps[(size_t)j * m + i] = acc[a][b][r];
      }
  }
}

// ---------------------------------------------------------------------------
// D = alpha A G + beta D.  Tiles of 128 rows x 32 NJ columns.  A lane holds
// the rows 2l, 2l + 1 of a 32-row group (one 16-byte LDS read), i.e. the real
// and imaginary part of one coefficient: two MFMA row blocks.  A's columns are
// copied straight to LDS (1 KiB each); G goes through registers, its 16-byte
// loads only where GV (even leading dimension, aligned).  M even; lda, ldd
// even and A, D 16-byte aligned.  INPL (D is A; G upper triangular, or all of n
// in one tile): a workgroup takes the column tiles of its rows from the last to
// the first, so that no column is written before every product that reads it.
// ---------------------------------------------------------------------------
template <int NJ, bool PROJ, bool GV, bool INPL>
__global__ __launch_bounds__(256, 2) void k_nn_f64(const double* A, int lda,
                                                   const double* __restrict__ G, int ldgm, int M, int k, int n,
                                                   double alpha, double beta, double* D, int ldd,
                                                   int upper_g, FnlEpi epi, ProjTab proj, int tn, int total) {
  constexpr int TI = 128, TJ = 32 * NJ;
  constexpr int kStageA = kKs * TI * 8, kStage = kStageA + TJ * 128;
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * kStage];
  const int t = xcd_index(total);
  if (t >= total) return;
  const int rt = INPL ? t : t / tn;
  const int i0 = rt * TI;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  for (int ct = INPL ? tn - 1 : t - rt * tn, left = INPL ? tn : 1; left > 0; --ct, --left) {
  if (INPL && left < tn) __syncthreads();   // the stages are free again
  const int j0 = ct * TJ;
  const int kmax = upper_g ? min(k, j0 + TJ) : k;
  // A: wave w copies the columns w, w + 4, ... of a slice; lane -> rows 2 lane,
  // 2 lane + 1.  Rows beyond M repeat the last pair: they are not stored.
  const int arow = min(i0 + 2 * lane, M - 2);
  d2 ea[4];
  double ta[4];
  int la[4];
  auto issue_a = [&](int kb, int st) {
    unsigned char* sa = lds + st * kStage;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int c = wave + 4 * u, kk = kb + c;
      if constexpr (PROJ) {   // (-i)^l twnl eigr of column kk (no gk: variant 0)
        const int4 c4 = proj.tab[kk];
        ea[u] = reinterpret_cast<const d2*>(proj.eigr)[(size_t)c4.x * proj.ldg + (arow >> 1)];
        ta[u] = proj.twnl[(size_t)c4.y * proj.ldg + (arow >> 1)];
        la[u] = c4.z;
      } else copy16_lds(A + (size_t)kk * lda + arow, (lds_void*)(sa + c * 1024));
    }
  };
  auto put_a = [&](int st) {
    if constexpr (PROJ) {
      unsigned char* sa = lds + st * kStage;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        *reinterpret_cast<d2*>(sa + (wave + 4 * u) * 1024 + lane * 16) = proj_value(Raw{ea[u], ta[u], 0.0}, la[u], false);
    }
  };
  // G: thread -> column t/8 + 32 u of the tile, k = 2 (t%8), + 1 of the slice.  Chunk
  // 4 h + q holds k = 8 h + q, 8 h + 4 + q: a 16-byte read feeds two instructions that
  // take four successive k each, the order of k_gemm_nn (same bits).
  const int gc = threadIdx.x >> 3, gq = threadIdx.x & 7;
  d2 rg[NJ];
  auto fetch_g = [&](int kb) {   // a whole slice; columns beyond n repeat the last one (not stored)
#pragma unroll
    for (int u = 0; u < NJ; ++u) {
      const double* src = G + (size_t)min(j0 + gc + 32 * u, n - 1) * ldgm + kb + 2 * gq;
      if constexpr (GV) rg[u] = *reinterpret_cast<const d2*>(src);
      else rg[u] = d2{src[0], src[1]};
    }
  };
  auto put_g = [&](int st) {
    unsigned char* sg = lds + st * kStage + kStageA;
#pragma unroll
    for (int u = 0; u < NJ; ++u) {
      double* d = reinterpret_cast<double*>(sg) + ((gq >> 1) & 1);
      const int q = (gq & 4) + 2 * (gq & 1);
      d[2 * chunk_slot(gc + 32 * u, q)] = rg[u].x;
      d[2 * chunk_slot(gc + 32 * u, q + 1)] = rg[u].y;
    }
  };
  const int wr = (wave >> 1) * 64, wc = (wave & 1) * 16 * NJ;
  const int li = lane & 15, lq = lane >> 4;
  d4 acc[2][2][NJ];   // [row group][row of the pair][column block]
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int b = 0; b < NJ; ++b) acc[a][p][b] = d4{0.0, 0.0, 0.0, 0.0};
  auto multiply = [&](int st) {
    const unsigned char* sa = lds + st * kStage;
    const unsigned char* sg = sa + kStageA;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      d2 fg[NJ];
#pragma unroll
      for (int b = 0; b < NJ; ++b)
        fg[b] = *reinterpret_cast<const d2*>(sg + 16 * chunk_slot(wc + 16 * b + li, 4 * h + lq));
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int kk = 8 * h + 4 * s + lq;
        d2 fa[2];
#pragma unroll
        for (int a = 0; a < 2; ++a)
          fa[a] = *reinterpret_cast<const d2*>(sa + kk * 1024 + (wr + 32 * a + 2 * li) * 8);
#pragma unroll
        for (int b = 0; b < NJ; ++b) {
          const double g = s ? fg[b].y : fg[b].x;
#pragma unroll
          for (int a = 0; a < 2; ++a) {
            acc[a][0][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(g, fa[a].x, acc[a][0][b], 0, 0, 0);
            acc[a][1][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(g, fa[a].y, acc[a][1][b], 0, 0, 0);
          }
        }
      }
    }
  };
  const int nfull = kmax / kKs;
  if (nfull > 0) {
    issue_a(0, 0);
    fetch_g(0);
    put_a(0);
    put_g(0);
  }
  int st = 0;
  for (int i = 0; i < nfull; ++i, st ^= 1) {
    slice_barrier();   // slice i is staged, and every wave is done with the other stage
    const bool more = i + 1 < nfull;
    if (more) {
      issue_a((i + 1) * kKs, st ^ 1);
      fetch_g((i + 1) * kKs);
    }
    multiply(st);
    if (more) {
      put_a(st ^ 1);
      put_g(st ^ 1);
    }
  }
  if (nfull * kKs < kmax) {   // the last columns of A, the rest of the slice zero
    unsigned char* sa = lds + st * kStage;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int c = wave + 4 * u, kk = nfull * kKs + c;
      d2 v = {0.0, 0.0};
      if (kk < kmax) {
        if constexpr (PROJ) {
          const ProjCol pc = proj_col(proj, kk);
          v = proj_value(proj_load(pc, arow >> 1), pc.l, false);
        } else {
          v = *reinterpret_cast<const d2*>(A + (size_t)kk * lda + arow);
        }
      }
      *reinterpret_cast<d2*>(sa + c * 1024 + lane * 16) = v;
    }
#pragma unroll
    for (int u = 0; u < NJ; ++u) {
      const int kk = nfull * kKs + 2 * gq;
      const double* src = G + (size_t)min(j0 + gc + 32 * u, n - 1) * ldgm + kk;
      rg[u] = d2{kk < kmax ? src[0] : 0.0, kk + 1 < kmax ? src[1] : 0.0};
    }
    put_g(st);
    __syncthreads();
    multiply(st);
  }
  // 16 lanes store 256 contiguous bytes of a column; four columns per register
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int i = i0 + wr + 32 * a + 2 * li;
    if (i >= M) continue;
    const double tw = !PROJ && epi.twnl ? epi.twnl[i >> 1] : 1.0;
#pragma unroll
    for (int b = 0; b < NJ; ++b) {
      double2 d[4];
      bool ok[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = j0 + wc + 16 * b + 4 * r + lq;
        ok[r] = j < n;
        if (ok[r] && beta != 0.0) d[r] = *reinterpret_cast<const double2*>(D + (size_t)j * ldd + i);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = j0 + wc + 16 * b + 4 * r + lq;
        if (!ok[r]) continue;
        const double x0 = acc[a][0][b][r], x1 = acc[a][1][b][r];
        double2 y;
        if (epi.f) {   // fnonloc: c2 -= f [(-i)^l twnl] (A G), f < 1e-5 -> 1
          double f = epi.f[j];
          if (f < 1e-5) f = 1.0;
          if constexpr (!PROJ) {
            f *= epi.lmod4 & 2 ? -tw : tw;
            y = epi.lmod4 & 1 ? make_double2(d[r].x - f * x1, d[r].y + f * x0)
                              : make_double2(d[r].x - f * x0, d[r].y - f * x1);
          } else {
            y = make_double2(d[r].x - f * x0, d[r].y - f * x1);
          }
        } else if (beta == 0.0) {
          y = make_double2(alpha * x0, alpha * x1);
        } else {
          y = make_double2(beta * d[r].x + alpha * x0, beta * d[r].y + alpha * x1);
        }
        *reinterpret_cast<double2*>(D + (size_t)j * ldd + i) = y;
        if constexpr (!PROJ) {
          if (epi.vcm) {
            const double2 c = *reinterpret_cast<const double2*>(A + (size_t)j * lda + i);
            *reinterpret_cast<double2*>(epi.vcm + (size_t)j * ldd + i) =
                make_double2(epi.vodt * (y.x - c.x), epi.vodt * (y.y - c.y));
          }
        }
      }
    }
  }
  }   // column tiles
}

// Cost of an edge of n in tiles of 32 w: the padded edge, narrow tiles
// counting for more (their workgroups stage more per product).
double edge_cost(int n, int w) { return (n + 32 * w - 1) / (32 * w) * (32.0 * w) * (1.0 + 0.3 / w); }

// The tile edge of least cost, in units of 32, from 1 to most (130 -> 5, 96 ->
// 3, 512 -> 4; the widest of equals)
int tile_width(int n, int least, int most) {
  int best = least;
  for (int w = least + 1; w <= most; ++w)
    if (edge_cost(n, w) <= edge_cost(n, best)) best = w;
  return best;
}

// Column tiles of A G out of place, 32 or 64 wide: the workgroups of wider ones
// fill the registers and LDS of a CU in twos, and nothing runs beside the first
// copies and the store of a tile, which count with the short K of most products
// here.  64 where there are 8 such tiles for each CU and the padding allows it.
// Widths 32, 64, 96, 128, 160 at M x k x n, us:
//   396,408 x 512 x 512   3628  3409  4037  3654  4462
//   136,700 x 512 x 130    232   258   272   348   300   (projectors)
//    26,100 x 386 x 512    198   227   252   231   275
//    13,050 x 512 x 386    115   111   113   145   171
//     1,900 x 128 x 128     16    17    22    27    32
int nn_width(int tm, int n) {
  const int w1 = (n + 31) / 32, w2 = (n + 63) / 64;
  return tm * (long long)w2 >= 2048 && w2 * 64 * 1.06 <= w1 * 32 * 1.12 ? 2 : 1;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <int NI, int NJ>
void launch_tn(mc_ctx* ctx, const double* A, int lda, const double* B, int ldb, int K, int m, int n, int kchunk,
               bool upper, const ProjTab* proj, int tm, int tn, int total) {
  const int launch = (total + kXcds - 1) / kXcds * kXcds;
  double* P = ctx->w_gemm.as<double>();
  if (!proj) {
    hipLaunchKernelGGL((k_tn_f64<NI, NJ, false>), dim3(launch), dim3(256), 0, ctx->stream, A, lda, B, ldb, K, m, n,
                       kchunk, P, upper ? 1 : 0, ProjTab{}, tm, tn, total);
  } else if constexpr (NI * NJ <= 16) {   // registers for the projector operand
    hipLaunchKernelGGL((k_tn_f64<NI, NJ, true>), dim3(launch), dim3(256), 0, ctx->stream, A, lda, B, ldb, K, m, n,
                       kchunk, P, upper ? 1 : 0, *proj, tm, tn, total);
  } else {
    throw Error{MC_ERR_INTERNAL, "projector tile too large"};
  }
}

template <int NI>
void launch_tn_j(int nj, mc_ctx* ctx, const double* A, int lda, const double* B, int ldb, int K, int m, int n,
                 int kchunk, bool upper, const ProjTab* proj, int tm, int tn, int total) {
  switch (nj) {
    case 1: launch_tn<NI, 1>(ctx, A, lda, B, ldb, K, m, n, kchunk, upper, proj, tm, tn, total); break;
    case 2: launch_tn<NI, 2>(ctx, A, lda, B, ldb, K, m, n, kchunk, upper, proj, tm, tn, total); break;
    case 3: launch_tn<NI, 3>(ctx, A, lda, B, ldb, K, m, n, kchunk, upper, proj, tm, tn, total); break;
    case 4: launch_tn<NI, 4>(ctx, A, lda, B, ldb, K, m, n, kchunk, upper, proj, tm, tn, total); break;
    default: launch_tn<NI, 5>(ctx, A, lda, B, ldb, K, m, n, kchunk, upper, proj, tm, tn, total); break;
  }
}

}  // namespace

bool tn_f64_form(const double* A, int lda, const double* B, int ldb) {
  return lda % 2 == 0 && ldb % 2 == 0 && aligned16(A) && aligned16(B);
}

// Partials of A^T B into ctx->w_gemm; returns their number.  proj: A is the
// projector operand of m columns (A, lda unused).  Where the device memory does not
// hold the partials, K is split less (with fewer); where it still does not, an error,
// or 0 for the projector operand.
int tn_f64_partials(mc_ctx* ctx, const double* A, int lda, const double* B, int ldb, int K, int m, int n,
                    bool symmetric, const ProjTab* proj, bool fewer) {
  const int mu = proj ? proj->ncol : m;   // rows that decide the tile and the split
  int ni = 2, nj = 1;
  if (symmetric) {   // square tiles
    ni = nj = n <= 64 ? 2 : tile_width(n, 3, 4);
  } else {
    double least = 0.0;
    for (int a = 2; a <= 4; ++a)
      for (int b = 1; b <= 5; ++b) {
        if (proj && a * b > 16) continue;
        const double c = edge_cost(proj ? 4 * mu : mu, a) * edge_cost(n, b);
        if (least == 0.0 || c <= least) {
          least = c;
          ni = a;
          nj = b;
        }
      }
  }
  if ((long long)((mu + 32 * ni - 1) / (32 * ni)) * ((n + 32 * nj - 1) / (32 * nj)) * (K / 128) < 256) {
    // too few tiles and K rows for a workgroup per CU: smaller tiles
    ni = 2;
    nj = symmetric ? 2 : tile_width(n, 1, 2);
  }
  const int tm = (m + 32 * ni - 1) / (32 * ni), tn = (n + 32 * nj - 1) / (32 * nj);
  const int tiles = tile_count(symmetric, tm, tn);
  // K chunks of at least 128 rows; the number of splits that fills whole rounds
  // of two workgroups per CU best (the fewest of equals), at most two rounds.
  // The projector products split K by one variant's columns (one round), so
  // that each variant's sums do not depend on which others are asked for.
  const int unit = proj ? (mu + 32 * ni - 1) / (32 * ni) * tn : tiles;
  const int most = std::max(1, std::min((proj ? 512 : 1024) / unit, K / 128));
  int nsplit = 1;
  double best = 0.0;
  for (int s = 1; s <= most; ++s) {
    const int w = s * unit, rounds = (w + 511) / 512;
    const double fill = w / (512.0 * rounds);
    if (fill > best + 1e-9) {
      best = fill;
      nsplit = s;
    }
  }
  int kchunk;
  for (;; nsplit /= 2) {
    kchunk = (K + nsplit - 1) / nsplit;
    kchunk = (kchunk + kKs - 1) / kKs * kKs;
    nsplit = (K + kchunk - 1) / kchunk;
    const bool last = nsplit == 1 || !fewer;
    if (try_ensure(ctx->w_gemm, sizeof(double) * (size_t)nsplit * m * n, last && !proj)) break;
    if (last) return 0;
  }
  const int total = nsplit * tiles;
  timer_begin(ctx, MC_KID_GEMM_TN);
  if (ni == 2)
    launch_tn_j<2>(nj, ctx, A, lda, B, ldb, K, m, n, kchunk, symmetric, proj, tm, tn, total);
  else if (ni == 3)
    launch_tn_j<3>(nj, ctx, A, lda, B, ldb, K, m, n, kchunk, symmetric, proj, tm, tn, total);
  else
    launch_tn_j<4>(nj, ctx, A, lda, B, ldb, K, m, n, kchunk, symmetric, proj, tm, tn, total);
  MC_HIP(hipGetLastError());
  timer_end(ctx, MC_KID_GEMM_TN);
  return nsplit;
}

bool nn_f64_form(const double* A, int lda, int M, const double* D, int ldd, const FnlEpi* epi) {
  return M >= 2 && M % 2 == 0 && lda % 2 == 0 && ldd % 2 == 0 && aligned16(A) && aligned16(D) &&
         (!epi || aligned16(epi->vcm));
}

bool nn_f64_in_place(int n, bool upper_g) { return upper_g || n <= 32 * tile_width(n, 1, 5); }

void nn_f64(mc_ctx* ctx, const double* A, int lda, const double* G, int ldgm, int M, int k, int n, double alpha,
            double beta, double* D, int ldd, bool upper_g, const FnlEpi& epi, const ProjTab* proj, int kid) {
  const bool inpl = D == A;
  const int tm = (M + 127) / 128;
  const int nj = inpl ? tile_width(n, 1, 5) : nn_width(tm, n);
  const int tn = (n + 32 * nj - 1) / (32 * nj);
  MC_CHECK(!inpl || nn_f64_in_place(n, upper_g), MC_ERR_INTERNAL, "A G in place needs an upper G or one column tile");
  const int total = inpl ? tm : tm * tn, launch = (total + kXcds - 1) / kXcds * kXcds;
  const bool gv = ldgm % 2 == 0 && aligned16(G);
  const ProjTab pt = proj ? *proj : ProjTab{};
  timer_begin(ctx, kid);
#define MC_NN(NJ, PR, GV, IP)                                                                                 \
  hipLaunchKernelGGL((k_nn_f64<NJ, PR, GV, IP>), dim3(launch), dim3(256), 0, ctx->stream, A, lda, G, ldgm, M, k, n, \
                     alpha, beta, D, ldd, upper_g ? 1 : 0, epi, pt, tn, total)
#define MC_NN_I(NJ)                            \
  do {                                         \
    if (gv) MC_NN(NJ, false, true, true);      \
    else MC_NN(NJ, false, false, true);        \
  } while (0)
#define MC_NN_J(NJ)                                    \
  do {                                                 \
    if (proj && gv) MC_NN(NJ, true, true, false);      \
    else if (proj) MC_NN(NJ, true, false, false);      \
    else if (gv) MC_NN(NJ, false, true, false);        \
    else MC_NN(NJ, false, false, false);               \
  } while (0)
  if (!inpl) {
    if (nj == 1) MC_NN_J(1);
    else MC_NN_J(2);
  } else {
    switch (nj) {
      case 1: MC_NN_I(1); break;
      case 2: MC_NN_I(2); break;
      case 3: MC_NN_I(3); break;
      case 4: MC_NN_I(4); break;
      default: MC_NN_I(5); break;
    }
  }
#undef MC_NN_J
#undef MC_NN_I
#undef MC_NN
  MC_HIP(hipGetLastError());
  timer_end(ctx, kid);
}

}  // namespace mc
