// Device-side 1D transforms for gfx950, templated on the arithmetic type
// (double for the FP64 path, float for the mixed-precision path).
//
// Sign convention (CPMD, src/mltfft_utils.mod.F90:513-517): the inverse
// transform (G -> r) is e^{+i 2 pi k x / n}, unscaled; the forward transform
// (r -> G) is e^{-i 2 pi k x / n}; the 1/(n1 n2 n3) scale is applied by the
// caller after the last forward pass.
//
// Three engines, all cooperative over one workgroup of kThreads threads on a
// batch of lines held in LDS (line stride `lds`):
//  * fft_fast<T, N, DIR>: lengths N = A*B known at compile time, two LDS round
//    trips per transform.  Four-step form (A, B <= 20): each thread does one
//    length-A DFT in registers over x[B n1 + n2] (stride B), multiplies by
//    w_N^{n2 k1}, the lines are transposed in LDS and each thread does one
//    length-B DFT in registers.  Register DFTs of composite length recurse at
//    compile time into radix 2/3/4/5/7 butterflies with exact constant twiddles
//    (twiddle_consts.h).  Stage form (FP32 at the lengths of MC_MORE_SIZES): the
//    stages of the runtime plan, grouped A and B <= 25 points at a time in registers.
//  * fft_lines<T, DIR>: any 2^a 3^b 5^c 7^d length from a runtime plan: mixed-radix
//    Stockham stages; stage s with radix R and p = product of previous radices
//    maps butterfly i of a line to inputs x[i + q n/R], twiddles w^{q k n/(pR)}
//    (k = i mod p) and outputs y[(i-k) R + k + s p], in place with two barriers.
#pragma once

#include <hip/hip_runtime.h>

#include "mc_internal.h"
#include "twiddle_consts.h"

namespace mc {

constexpr int kThreads = 256;   // threads per workgroup of every transform kernel
constexpr int kMaxBfly = 4;     // butterflies per thread and stage (generic engine)

template <typename T> struct V2;
template <> struct V2<double> { using type = double2; };
template <> struct V2<float> { using type = float2; };
template <typename T> using v2 = typename V2<T>::type;

template <typename V>
__device__ __forceinline__ V cadd(V a, V b) { V r; r.x = a.x + b.x; r.y = a.y + b.y; return r; }
template <typename V>
__device__ __forceinline__ V csub(V a, V b) { V r; r.x = a.x - b.x; r.y = a.y - b.y; return r; }
template <typename V>
__device__ __forceinline__ V cscale(V a, decltype(a.x) s) { V r; r.x = a.x * s; r.y = a.y * s; return r; }
template <typename V>
__device__ __forceinline__ V cmk(decltype(V().x) x, decltype(V().x) y) { V r; r.x = x; r.y = y; return r; }

// a * w when DIR < 0 (forward), a * conj(w) when DIR > 0 (inverse); w = exp(-2 pi i t/n)
template <int DIR, typename V>
__device__ __forceinline__ V twmul(V a, V w) {
  if (DIR < 0) return cmk<V>(a.x * w.x - a.y * w.y, a.x * w.y + a.y * w.x);
  return cmk<V>(a.x * w.x + a.y * w.y, a.y * w.x - a.x * w.y);
}
// a * DIR * i
template <int DIR, typename V>
__device__ __forceinline__ V mul_di(V a) {
  if (DIR < 0) return cmk<V>(a.y, -a.x);
  return cmk<V>(-a.y, a.x);
}

// ---------------------------------------------------------------------------
// radix butterflies in registers
// ---------------------------------------------------------------------------
template <int DIR, typename V>
__device__ __forceinline__ void bfly2(V* v) {
  V a = v[0], b = v[1];
  v[0] = cadd(a, b); v[1] = csub(a, b);
}
template <int DIR, typename V>
__device__ __forceinline__ void bfly4(V* v) {
  V t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
  V t2 = cadd(v[1], v[3]), t3 = mul_di<DIR>(csub(v[1], v[3]));
  v[0] = cadd(t0, t2); v[2] = csub(t0, t2);
  v[1] = cadd(t1, t3); v[3] = csub(t1, t3);
}
template <int DIR, typename V>
__device__ __forceinline__ void bfly3(V* v) {
  using T = decltype(V().x);
  const T s3 = (T)0.86602540378443864676;   // sin(2 pi/3)
  V t1 = cadd(v[1], v[2]);
  V t2 = csub(v[1], v[2]);
  V y0 = cadd(v[0], t1);
  V m = cmk<V>(v[0].x - (T)0.5 * t1.x, v[0].y - (T)0.5 * t1.y);
  V r = mul_di<DIR>(cscale(t2, s3));
  v[0] = y0; v[1] = cadd(m, r); v[2] = csub(m, r);
}
template <int DIR, typename V>
__device__ __forceinline__ void bfly5(V* v) {
  using T = decltype(V().x);
  const T c1 = (T)0.30901699437494742410;    // cos(2 pi/5)
  const T c2 = (T)-0.80901699437494742410;   // cos(4 pi/5)
  const T s1 = (T)0.95105651629515357212;    // sin(2 pi/5)
  const T s2 = (T)0.58778525229247312917;    // sin(4 pi/5)
  V t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]);
  V t3 = csub(v[1], v[4]), t4 = csub(v[2], v[3]);
  V y0 = cadd(v[0], cadd(t1, t2));
  V a1 = cmk<V>(v[0].x + c1 * t1.x + c2 * t2.x, v[0].y + c1 * t1.y + c2 * t2.y);
  V a2 = cmk<V>(v[0].x + c2 * t1.x + c1 * t2.x, v[0].y + c2 * t1.y + c1 * t2.y);
  V b1 = mul_di<DIR>(cmk<V>(s1 * t3.x + s2 * t4.x, s1 * t3.y + s2 * t4.y));
  V b2 = mul_di<DIR>(cmk<V>(s2 * t3.x - s1 * t4.x, s2 * t3.y - s1 * t4.y));
  v[0] = y0;
  v[1] = cadd(a1, b1); v[4] = csub(a1, b1);
  v[2] = cadd(a2, b2); v[3] = csub(a2, b2);
}

// 7-point DFT: t_k = v_k + v_{7-k}, u_k = v_k - v_{7-k} (k = 1..3);
// y_m = v_0 + sum_k cos(2 pi k m/7) t_k + DIR i sum_k sin(2 pi k m/7) u_k and
// y_{7-m} with the sine term negated (m = 1..3)
template <int DIR, typename V>
__device__ __forceinline__ void bfly7(V* v) {
  using T = decltype(V().x);
  V t[3], u[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    t[k] = cadd(v[k + 1], v[6 - k]);
    u[k] = csub(v[k + 1], v[6 - k]);
  }
  const V x0 = v[0];
  v[0] = cadd(x0, cadd(t[0], cadd(t[1], t[2])));
#pragma unroll
  for (int m = 1; m <= 3; ++m) {
    V a = x0, b = cmk<V>((T)0, (T)0);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int j = ((k + 1) * m) % 7;
      const T c = (T)TwC<7>::c[j], s = (T)TwC<7>::s[j];
      a = cmk<V>(a.x + c * t[k].x, a.y + c * t[k].y);
      b = cmk<V>(b.x + s * u[k].x, b.y + s * u[k].y);
    }
    b = mul_di<DIR>(b);
    v[m] = cadd(a, b);
    v[7 - m] = csub(a, b);
  }
}

template <int R>
struct Split {   // R = P * Q for the register recursion
  static constexpr int P = (R % 4 == 0 && R != 4) ? 4
                           : (R % 3 == 0 && R != 3) ? 3
                           : (R % 2 == 0 && R != 2) ? 2
                           : (R % 5 == 0 && R != 5) ? 5
                                                    : 7;
  static constexpr int Q = R / P;
};

// v[j] *= W_R^e (DIR < 0) or conj (DIR > 0), e compile-time
template <int R, int DIR, typename V>
__device__ __forceinline__ V twc(V a, int e) {
  using T = decltype(V().x);
  const T c = (T)TwC<R>::c[e], s = (T)TwC<R>::s[e];
  // W = c - i s
  if (DIR < 0) return cmk<V>(a.x * c + a.y * s, a.y * c - a.x * s);
  return cmk<V>(a.x * c - a.y * s, a.y * c + a.x * s);
}

// in-register DFT of length R: v[k] <- sum_n v[n] w^{DIR n k}
template <int R, int DIR, typename V>
__device__ __forceinline__ void dftn(V* v) {
  if constexpr (R == 1) {
    return;
  } else if constexpr (R == 2) {
    bfly2<DIR>(v);
  } else if constexpr (R == 3) {
    bfly3<DIR>(v);
  } else if constexpr (R == 4) {
    bfly4<DIR>(v);
  } else if constexpr (R == 5) {
    bfly5<DIR>(v);
  } else if constexpr (R == 7) {
    bfly7<DIR>(v);
  } else {
    constexpr int P = Split<R>::P, Q = Split<R>::Q;
    V y[R];
#pragma unroll
    for (int n2 = 0; n2 < Q; ++n2) {
      V u[P];
#pragma unroll
      for (int n1 = 0; n1 < P; ++n1) u[n1] = v[Q * n1 + n2];
      dftn<P, DIR>(u);
#pragma unroll
      for (int k1 = 0; k1 < P; ++k1) y[n2 * P + k1] = ((n2 * k1) % R == 0) ? u[k1] : twc<R, DIR>(u[k1], (n2 * k1) % R);
    }
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) {
      V u[Q];
#pragma unroll
      for (int n2 = 0; n2 < Q; ++n2) u[n2] = y[n2 * P + k1];
      dftn<Q, DIR>(u);
#pragma unroll
      for (int k2 = 0; k2 < Q; ++k2) v[k1 + P * k2] = u[k2];
    }
  }
}

// 16-point register DFT for the band of the wavefunction sphere (frequencies
// |m| < N/4 of an N = 16 B transform sit at k = 0..3 and 12..15 of the
// four-step's 16-point DFTs).  IN: the inputs 4..11 are zero and not read
// (the first radix-4 stage reduces to a +- d, a -+ DIR i d); OUT: only the
// outputs 0..3 and 12..15 are formed (4..11 keep what they held).  On the
// entries it forms it does dftn<16>'s arithmetic, so the values agree with it
// (up to the sign of zero results).
template <int DIR, bool IN, bool OUT, typename V>
__device__ __forceinline__ void dft16_band(V* v) {
  V y[16];
#pragma unroll
  for (int n2 = 0; n2 < 4; ++n2) {
    V u[4];
    if constexpr (IN) {
      const V a = v[n2], d = v[12 + n2];
      const V md = mul_di<DIR>(d);
      u[0] = cadd(a, d);
      u[1] = csub(a, md);
      u[2] = csub(a, d);
      u[3] = cadd(a, md);
    } else {
#pragma unroll
      for (int n1 = 0; n1 < 4; ++n1) u[n1] = v[4 * n1 + n2];
      bfly4<DIR>(u);
    }
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) y[n2 * 4 + k1] = ((n2 * k1) % 16 == 0) ? u[k1] : twc<16, DIR>(u[k1], (n2 * k1) % 16);
  }
#pragma unroll
  for (int k1 = 0; k1 < 4; ++k1) {
    V u[4];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) u[n2] = y[n2 * 4 + k1];
    if constexpr (OUT) {
      const V t0 = cadd(u[0], u[2]), t1 = csub(u[0], u[2]);
      const V t2 = cadd(u[1], u[3]), t3 = mul_di<DIR>(csub(u[1], u[3]));
      v[k1] = cadd(t0, t2);
      v[k1 + 12] = csub(t1, t3);
    } else {
      bfly4<DIR>(u);
#pragma unroll
      for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = u[k2];
    }
  }
}

// As dft16_band<DIR, true, false> for any A = 4 Q: the inputs Q .. 3Q - 1 are
// zero and not read.
template <int A, int DIR, typename V>
__device__ __forceinline__ void dft_band_in(V* v) {
  constexpr int Q = A / 4;
  static_assert(A % 4 == 0 && A > 4, "band DFT of a length 4 Q");
  V y[A];
#pragma unroll
  for (int n2 = 0; n2 < Q; ++n2) {
    const V a = v[n2], d = v[3 * Q + n2];
    const V md = mul_di<DIR>(d);
    const V u[4] = {cadd(a, d), csub(a, md), csub(a, d), cadd(a, md)};
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) y[n2 * 4 + k1] = ((n2 * k1) % A == 0) ? u[k1] : twc<A, DIR>(u[k1], (n2 * k1) % A);
  }
#pragma unroll
  for (int k1 = 0; k1 < 4; ++k1) {
    V u[Q];
#pragma unroll
    for (int n2 = 0; n2 < Q; ++n2) u[n2] = y[n2 * 4 + k1];
    dftn<Q, DIR>(u);
#pragma unroll
    for (int k2 = 0; k2 < Q; ++k2) v[k1 + 4 * k2] = u[k2];
  }
}

// ---------------------------------------------------------------------------
// compile-time four-step engine
// ---------------------------------------------------------------------------
template <int N> struct FastShape { static constexpr int A = 0, B = 0; };
#define MC_FAST_SHAPE(n, a, b) \
  template <> struct FastShape<n> { static constexpr int A = a, B = b; };
MC_FAST_SHAPE(16, 4, 4)
MC_FAST_SHAPE(18, 6, 3)
MC_FAST_SHAPE(24, 6, 4)
MC_FAST_SHAPE(54, 9, 6)
MC_FAST_SHAPE(128, 16, 8)
MC_FAST_SHAPE(192, 16, 12)
MC_FAST_SHAPE(224, 16, 14)
MC_FAST_SHAPE(240, 16, 15)
MC_FAST_SHAPE(30, 6, 5)
MC_FAST_SHAPE(32, 8, 4)
MC_FAST_SHAPE(36, 6, 6)
MC_FAST_SHAPE(40, 8, 5)
MC_FAST_SHAPE(48, 8, 6)
MC_FAST_SHAPE(60, 10, 6)
MC_FAST_SHAPE(64, 8, 8)
MC_FAST_SHAPE(72, 8, 9)
MC_FAST_SHAPE(80, 8, 10)
MC_FAST_SHAPE(90, 10, 9)
MC_FAST_SHAPE(96, 12, 8)
MC_FAST_SHAPE(100, 10, 10)
MC_FAST_SHAPE(108, 12, 9)
MC_FAST_SHAPE(120, 12, 10)
MC_FAST_SHAPE(144, 12, 12)
MC_FAST_SHAPE(150, 15, 10)
MC_FAST_SHAPE(160, 16, 10)
MC_FAST_SHAPE(162, 18, 9)
MC_FAST_SHAPE(180, 12, 15)
MC_FAST_SHAPE(200, 20, 10)
MC_FAST_SHAPE(216, 12, 18)
MC_FAST_SHAPE(256, 16, 16)
MC_FAST_SHAPE(270, 18, 15)
MC_FAST_SHAPE(288, 16, 18)
MC_FAST_SHAPE(300, 20, 15)
MC_FAST_SHAPE(320, 16, 20)
#undef MC_FAST_SHAPE
// The lengths with a compile-time engine.  The second list is the rest of
// CPMD's even default lengths from 30 to 320, i.e. the meshes of cells of any
// edge, with factors A = 4 Q where the two stay close (band pruning).  The
// runtime-plan engine divides by runtime lengths for every butterfly and passes
// through LDS three to five times: density of 103 states on 108 x 120 x 160 in
// FP64 0.58 against 3.69 ms, gradient of 61 states on 80 x 144 x 96 with FP32
// transforms 0.36 against 1.08 ms.
#define MC_FAST_SIZES(X) X(16) X(18) X(24) X(54) X(128) X(192) X(224) X(240)
#define MC_MORE_SIZES(X)                                                                                    \
  X(30) X(32) X(36) X(40) X(48) X(60) X(64) X(72) X(80) X(90) X(96) X(100) X(108) X(120) X(144) X(150) X(160) \
  X(162) X(180) X(200) X(216) X(256) X(270) X(288) X(300) X(320)

// The radices of the runtime plan (make_plan) of length N, and the split A B of
// its stages that stays closest: A the product of the first stages, radix 5 left
// to the second group (100 = 20 x 5 does not round as the plan's kernels do, 4 x
// 25 does)
struct StageList {
  int nf = 0;
  int rad[kMaxStages] = {};
};
constexpr StageList stage_list(int n) {
  StageList s;
  for (int r : {4, 2, 3, 5, 7})
    while (n % r == 0) {
      s.rad[s.nf++] = r;
      n /= r;
    }
  return s;
}
constexpr int stage_split(int n) {
  const StageList s = stage_list(n);
  int best = 1, p = 1;
  for (int i = 0; i < s.nf; ++i) {
    p *= s.rad[i];
    if (s.rad[i] == 5) break;
    const int cur = best > n / best ? best : n / best, now = p > n / p ? p : n / p;
    if (now <= cur) best = p;
  }
  return best;
}

// Which compile-time engine length N has: the four-step one (FP64, and FP32 at
// the lengths of MC_FAST_SIZES) or, in FP32 at the others, the stages of the
// runtime plan two groups at a time in registers (stock_stages): the same
// operations on the same values in the same order.  Run beside the runtime plan's
// kernels at each of these lengths on each axis, with and without pruning, vpsi had
// the same bits everywhere, and rho those bits up to the last places of the FP64
// charge sums that scale it.  That rests on which products the compiler fuses
// (twmul_stage, stage_end) and can change with it: the tests hold FP32's 2e-6.
template <typename T, int N>
constexpr bool four_step() {
  if (sizeof(T) == 8) return true;
#define MC_CASE(x) if (N == x) return true;
  MC_FAST_SIZES(MC_CASE)
#undef MC_CASE
  return false;
}
template <typename T, int N>
struct Shape {
  static constexpr int A = four_step<T, N>() ? FastShape<N>::A : stage_split(N);
  static constexpr int B = N / A;
};

// Keeps the compiler from merging arithmetic across this point (no
// instruction): the runtime plan stores to LDS between its stages, and a product
// or sum combined or vectorised across a stage boundary rounds differently.
__device__ __forceinline__ void stage_end(float2& v) { asm("" : "+v"(v.x), "+v"(v.y)); }

// twmul with the products that the compiler fuses in the runtime plan's kernels
// written out: left to it, vectorised code fuses the other ones
template <int DIR>
__device__ __forceinline__ float2 twmul_stage(float2 a, float2 w) {
  if (DIR < 0)
    return make_float2(__builtin_fmaf(a.x, w.x, -(a.y * w.y)), __builtin_fmaf(a.y, w.x, a.x * w.y));
  return make_float2(__builtin_fmaf(a.x, w.x, a.y * w.y), __builtin_fmaf(a.y, w.x, -(a.x * w.y)));
}

// Stages [S0, S0 + ...) of the runtime plan on the A (or B) values one thread
// holds: v of length LEN, local product P of the stages done here, p = P * K
// overall with this thread's k = k0 + K (0 .. P-1); tw: the N-point table.
// IN (first stage a radix 4): the values LEN/4 .. 3 LEN/4 - 1 are zero and not read.
template <int N, int S, int LEN, int P, int K, int DIR, bool IN, typename V>
__device__ __forceinline__ void stock_stages(V* v, int k0, const V* tw) {
  if constexpr (P < LEN) {
    constexpr int R = stage_list(N).rad[S];
    constexpr int M = LEN / (P * R);
    static_assert(LEN % (P * R) == 0, "stages of the group");
    V y[LEN];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int kk = 0; kk < P; ++kk) {
        V u[R];
        if constexpr (IN && P == 1) {
          static_assert(R == 4, "band of a radix-4 first stage");
          const V a = v[m], d = v[m + 3 * M];
          const V md = mul_di<DIR>(d);
          u[0] = cadd(a, d);
          u[1] = csub(a, md);
          u[2] = csub(a, d);
          u[3] = cadd(a, md);
        } else {
#pragma unroll
          for (int q = 0; q < R; ++q) u[q] = v[(m + q * M) * P + kk];
          if constexpr (P * K > 1) {
            const int k = k0 + K * kk;
            if (K > 1 || kk > 0) {
#pragma unroll
              for (int q = 1; q < R; ++q) u[q] = twmul_stage<DIR>(u[q], tw[q * k * (N / (P * K * R))]);
            }
          }
          dftn<R, DIR>(u);
        }
#pragma unroll
        for (int q = 0; q < R; ++q) y[m * P * R + kk + q * P] = u[q];
      }
#pragma unroll
    for (int i = 0; i < LEN; ++i) {
      v[i] = y[i];
      stage_end(v[i]);
    }
    stock_stages<N, S + 1, LEN, P * R, K, DIR, IN, V>(v, k0, tw);
  }
}
// index of the first stage of the second group
template <int N, int A>
constexpr int second_stage() {
  const StageList s = stage_list(N);
  int p = 1, i = 0;
  while (p < A) p *= s.rad[i++];
  return i;
}

// In-place transform of `nlines` lines (line stride lds) with tw = LDS copy of
// the N-point table; nlines * max(A, B) <= kThreads.  Begins and ends with a barrier
// point (callers synchronise before, this returns after a __syncthreads).
template <typename T, int N, int DIR>
__device__ __forceinline__ void fft_fast(v2<T>* buf, int nlines, int lds, const v2<T>* tw) {
  using V = v2<T>;
  constexpr int A = Shape<T, N>::A, B = Shape<T, N>::B;
  static_assert(A * B == N && A >= 1 && B >= 1, "unsupported fast length");
  V v[A];
  const int t = threadIdx.x;
  // step 1: thread (line, n2) transforms x[B n1 + n2], n1 < A
  const bool act1 = t < nlines * B;
  const int l1 = act1 ? t / B : 0, n2 = act1 ? t - l1 * B : 0;
  V* x1 = buf + l1 * lds;
  if (act1) {
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) v[n1] = x1[B * n1 + n2];
    if constexpr (four_step<T, N>()) {
      dftn<A, DIR>(v);
#pragma unroll
      for (int k1 = 1; k1 < A; ++k1) v[k1] = twmul<DIR>(v[k1], tw[n2 * k1]);
    } else {
      stock_stages<N, 0, A, 1, 1, DIR, false>(v, 0, tw);
    }
  }
  __syncthreads();
  if (act1) {
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) x1[k1 * B + n2] = v[k1];
  }
  __syncthreads();
  // step 2: thread (line, k1) transforms y[n2][k1], n2 < B
  const bool act2 = t < nlines * A;
  const int l2 = act2 ? t / A : 0, k1 = act2 ? t - l2 * A : 0;
  V* x2 = buf + l2 * lds;
  V u[B];
  if (act2) {
#pragma unroll
    for (int m = 0; m < B; ++m) u[m] = x2[k1 * B + m];
    if constexpr (four_step<T, N>()) dftn<B, DIR>(u);
    else stock_stages<N, second_stage<N, A>(), B, 1, A, DIR, false>(u, k1, tw);
  }
  __syncthreads();
  if (act2) {
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) x2[k1 + A * k2] = u[k2];
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------
// runtime-plan Stockham engine
// ---------------------------------------------------------------------------
template <int R, int DIR, typename V>
__device__ __forceinline__ void fft_stage(V* buf, int nlines, int lds, int n, int p, const V* tw) {
  const int nb = n / R;
  const int total = nlines * nb;
  const int tstride = n / (p * R);
  V v[kMaxBfly][R];
  int dst[kMaxBfly];
#pragma unroll
  for (int t = 0; t < kMaxBfly; ++t) {
    const int b = threadIdx.x + t * kThreads;
    dst[t] = -1;
    if (b < total) {
      const int line = b / nb;
      const int i = b - line * nb;
      const int k = i % p;
      V* x = buf + line * lds;
#pragma unroll
      for (int q = 0; q < R; ++q) v[t][q] = x[i + q * nb];
      if (p > 1) {
#pragma unroll
        for (int q = 1; q < R; ++q) v[t][q] = twmul<DIR>(v[t][q], tw[q * k * tstride]);
      }
      dftn<R, DIR>(v[t]);
      dst[t] = line * lds + (i - k) * R + k;
    }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < kMaxBfly; ++t) {
    if (dst[t] >= 0) {
#pragma unroll
      for (int q = 0; q < R; ++q) buf[dst[t] + q * p] = v[t][q];
    }
  }
  __syncthreads();
}

template <typename T, int DIR>
__device__ void fft_lines(v2<T>* buf, int nlines, int lds, const FftPlan& pl, const v2<T>* tw) {
  int p = 1;
  for (int s = 0; s < pl.nf; ++s) {
    const int R = pl.rad[s];
    if (R == 4) fft_stage<4, DIR>(buf, nlines, lds, pl.n, p, tw);
    else if (R == 2) fft_stage<2, DIR>(buf, nlines, lds, pl.n, p, tw);
    else if (R == 3) fft_stage<3, DIR>(buf, nlines, lds, pl.n, p, tw);
    else if (R == 5) fft_stage<5, DIR>(buf, nlines, lds, pl.n, p, tw);
    else fft_stage<7, DIR>(buf, nlines, lds, pl.n, p, tw);
    p *= R;
  }
}

// one entry for both engines: N > 0 compile-time length, N == 0 runtime plan
template <typename T, int N, int DIR>
__device__ __forceinline__ void fft_any(v2<T>* buf, int nlines, int lds, const FftPlan& pl, const v2<T>* tw) {
  if constexpr (N > 0) fft_fast<T, N, DIR>(buf, nlines, lds, tw);
  else fft_lines<T, DIR>(buf, nlines, lds, pl, tw);
}

// Largest number of lines of length n one workgroup may transform at once (generic engine).
inline int max_lines(const FftPlan& pl) {
  int rmin = 5;
  for (int s = 0; s < pl.nf; ++s) rmin = pl.rad[s] < rmin ? pl.rad[s] : rmin;
  return (kMaxBfly * kThreads * rmin) / pl.n;
}

// Host side: lanes per line of the compile-time engine of length n (its larger
// factor; 0 when n has none).
template <typename T>
inline int fast_a(int n) {
#define MC_CASE(x) case x: return Shape<T, x>::A > Shape<T, x>::B ? Shape<T, x>::A : Shape<T, x>::B;
  switch (n) {
    MC_FAST_SIZES(MC_CASE)
    MC_MORE_SIZES(MC_CASE)
    default: return 0;
  }
#undef MC_CASE
}

}  // namespace mc
