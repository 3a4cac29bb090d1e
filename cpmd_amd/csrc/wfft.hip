// rhoofr and vpsi on gfx950: the stick-sparse 3D transforms of Gamma state
// pairs, fused with the wavefunction pack, the |psi|^2 accumulation, the
// V(r) multiply and the Gamma decode + kinetic term.
//
// Per batch of P state pairs the data path through HBM is
//   zinv : C0 runs (stick order)  -> sticks  A[pair][slot][z]       (pack + z^-1)
//   yinv : A                       -> columns B[pair][z][col][y]     (y^-1)
//   xrho : B (all P pairs)         -> rho(r)  (x^-1, |psi|^2, rho read/written once per batch)
//   xvpsi: B (all P pairs), V(r)   -> B       (x^-1, *V, x^+1; V read once per batch)
//   yfwd : B                       -> A       (y^+1)
//   zfwd : A, C0, C2               -> C2      (z^+1, 1/(n1 n2 n3), decode, kinetic, c2 +=)
// Every kernel is templated on the arithmetic type T of the transforms and of
// the A/B workspaces (double: FP64 path; float: mixed-precision path; C0, C2,
// V and rho stay FP64 in HBM) and on the compile-time length N of its axis
// (0 = runtime plan).
// Reference: vpsi src/vpsi_utils.mod.F90:376-675 (one pair per iteration through
// invfftn/fwfftn, src/fftmain_utils.mod.F90:71-157) and rhoofr
// src/rhoofr_utils.mod.F90:305-409.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <optional>
#include <string>
#include <vector>

#include "wfft_passes.h"

namespace mc {

__global__ void k_scale(double* __restrict__ x, size_t n, double v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    x[i] *= v;
}

__global__ void k_fill(double* __restrict__ x, size_t n, double v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    x[i] = v;
}

// The sums that rhoofr reads back, in one launch and in a fixed order (one
// thread per pair and sum took 33 us at 103 states on 108 x 120 x 160, this 4).  Workgroup
// p < npairs: the zinv partials red[(p gx + b) 4 + k] of pair p, k = 0..3, into
// out[4 p + k]; the other nsum workgroups: partial sums of rho[0..n) into out[4
// npairs + ..].
__global__ __launch_bounds__(kThreads) void k_rho_sums(const double* __restrict__ red, int gx, int npairs,
                                                       const double* __restrict__ rho, size_t n, int nsum,
                                                       double* __restrict__ out) {
  __shared__ double part[kThreads];
  if ((int)blockIdx.x < npairs) {
    const int p = blockIdx.x, k = threadIdx.x & 3;
    double s = 0.0;
    for (int b = threadIdx.x >> 2; b < gx; b += kThreads / 4) s += red[((size_t)p * gx + b) * 4 + k];
    part[threadIdx.x] = s;
    __syncthreads();
    for (int h = kThreads / 2; h >= 4; h >>= 1) {
      if ((int)threadIdx.x < h) part[threadIdx.x] += part[threadIdx.x + h];
      __syncthreads();
    }
    if (threadIdx.x < 4) out[(size_t)p * 4 + threadIdx.x] = part[threadIdx.x];
    return;
  }
  const int q = blockIdx.x - npairs;
  double s = 0.0;
  for (size_t i = q * (size_t)kThreads + threadIdx.x; i < n; i += (size_t)nsum * kThreads) s += rho[i];
  s = warp_sum(s);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int v = 0; v < kThreads / 64; ++v) t += part[v];
    out[(size_t)4 * npairs + q] = t;
  }
}

// ---------------------------------------------------------------------------
// host drivers
// ---------------------------------------------------------------------------
static WParams make_params(mc_ctx* ctx) {
  WParams w;
  w.n1 = ctx->n1; w.n2 = ctx->n2; w.n3 = ctx->n3;
  w.kr1 = ctx->kr1; w.kr2 = ctx->kr2; w.kr3 = ctx->kr3;
  w.ngw = ctx->ngw; w.ldg = ctx->ldg; w.n_own = ctx->n_own; w.n_slots = ctx->n_slots;
  w.ncols = ctx->ncols; w.geq0 = ctx->geq0;
  w.tpiba2 = ctx->tpiba2; w.omega = ctx->omega;
  w.p1 = ctx->plan1; w.p2 = ctx->plan2; w.p3 = ctx->plan3;
  w.ginfo = ctx->d_ginfo.as<int>();
  w.hg = ctx->d_hg.as<double>();
  w.own_start = ctx->d_own_start.as<int>();
  w.col_start = ctx->d_col_start.as<int>();
  w.col_slot = ctx->d_col_slot.as<int>();
  w.col_gy = ctx->d_col_gy.as<int>();
  w.col_gx = ctx->d_col_gx.as<int>();
  w.tw1 = ctx->d_tw1.as<double2>();
  w.tw2 = ctx->d_tw2.as<double2>();
  w.tw3 = ctx->d_tw3.as<double2>();
  return w;
}

template <typename T>
static Shapes shapes(mc_ctx* ctx) {
  Shapes s;
  MC_CHECK(lines_for<T>(ctx->plan3) >= 2, MC_ERR_UNSUPPORTED, "nr3 too large for the z pass");
  s.lo = lines_for<T>(ctx->plan3) / 2;
  s.tz = lines_for<T>(ctx->plan2);
  s.ty = std::min(lines_for<T>(ctx->plan1), (kMaxElem * kThreads) / ctx->n1);
  s.ty = std::min(s.ty, (kMaxCol * kThreads) / std::max(ctx->ncols, 1));
  MC_CHECK(s.ty >= 1, MC_ERR_UNSUPPORTED, "nr1 too large for the x pass");
  s.gx = (ctx->n_own + s.lo - 1) / s.lo;
  // FP32 zfwd runs half as many sticks per workgroup as zinv.  Measured per
  // 128-pair launch at 192^3: zfwd 0.28 ms at 4 sticks against 0.31 ms at 8,
  // zinv 0.52 ms at 4 against 0.46 ms at 8
  s.lf = sizeof(T) == 4 ? std::max(1, s.lo / 2) : s.lo;
  s.gf = (ctx->n_own + s.lf - 1) / s.lf;
  return s;
}

// Pairs per transform batch: at most P, and under a device memory limit as
// many as fit beside everything else the library holds and a reserve for the
// buffers the rest of a step allocates after the transforms (vofrho's dense
// mesh, contraction partials: max(256 MiB, limit / 16)); the workspaces are
// shrunk when they hold more; MC_ERR_ARG when not even one pair fits.  A later
// allocation that still does not fit frees them while they are idle
// (ws_reclaim), and the next transform call sizes them again.
template <typename T>
static int fit_pairs(mc_ctx* ctx, int P, size_t extra) {
  const size_t lim = mem_limit();
  if (!lim) return P;
  const size_t per = sizeof(v2<T>) * ((size_t)ctx->n_slots * ctx->n3 + (size_t)ctx->n3 * ctx->ncols * ctx->n2);
  const size_t held = ctx->w_a.bytes + ctx->w_b.bytes;
  const size_t reserve = std::max((size_t)256 << 20, lim / 16);
  const size_t others = mem_current() - std::min(held, mem_current()) + extra + reserve;
  const size_t avail = lim > others ? lim - others : 0;
  const long long fit = (long long)(avail / per);
  if (fit < 1)
    throw Error{MC_ERR_ARG, "device memory limit of " + std::to_string(lim) + " bytes leaves " +
                                std::to_string(avail) + " bytes for the transform workspaces; one state pair needs " +
                                std::to_string(per)};
  if (fit < P) P = (int)fit;
  if (held > (size_t)P * per) {   // shrink to what the batch needs
    ctx->w_a.release();
    ctx->w_b.release();
  }
  return P;
}

template <typename T>
static void ensure_workspace(mc_ctx* ctx, int P, bool need_b = true) {
  ctx->w_a.ensure(sizeof(v2<T>) * (size_t)P * ctx->n_slots * ctx->n3);
  if (need_b) ctx->w_b.ensure(sizeof(v2<T>) * (size_t)P * ctx->n3 * ctx->ncols * ctx->n2);
}

// Column reuse: the columns of all npairs pairs in w_keep, when reuse is on,
// no device memory limit is set and the allocation succeeds (else nullptr:
// the caller works in batches as usual)
template <typename T>
static v2<T>* keep_columns(mc_ctx* ctx, int npairs) {
  if (!ctx->col_reuse || mem_limit() != 0 || npairs <= 0) return nullptr;
  const size_t bytes = sizeof(v2<T>) * (size_t)npairs * ctx->n3 * ctx->ncols * ctx->n2;
  return try_ensure(ctx->w_keep, bytes) ? ctx->w_keep.as<v2<T>>() : nullptr;
}

static void upload_f(mc_ctx* ctx, const double* f_host, int nstate) {
  ctx->w_f.ensure(sizeof(double) * std::max(nstate, 1));
  if (nstate)
    MC_HIP(hipMemcpyAsync(ctx->w_f.p, f_host, sizeof(double) * nstate, hipMemcpyHostToDevice, ctx->stream));
}

template <typename T>
static void rhoofr_impl(mc_ctx* ctx, const double2* c0, const double* f_host, int nstate, double* rho,
                        double* ekin, double* csumg, double* csumr, bool keep) {
  using V = v2<T>;
  const size_t nnr1 = (size_t)ctx->kr1 * ctx->kr2 * ctx->kr3;
  const WParams w = make_params(ctx);
  const Shapes s = shapes<T>(ctx);
  const int npairs = (nstate + 1) / 2;
  const int nblk_sum = (int)std::min<size_t>(1024, (nnr1 + 2047) / 2048);
  WsUse use(ctx->w_a, ctx->w_b);
  ctx->keep_valid = false;
  V* K = keep ? keep_columns<T>(ctx, npairs) : nullptr;
  std::optional<WsUse> use_keep;
  if (K)
    use_keep.emplace(ctx->w_keep, ctx->w_keep);
  else if (mem_limit() != 0)
    ctx->w_keep.release();   // stale columns: room for the batch workspaces
  const size_t red_bytes =
      sizeof(double) * ((size_t)std::max(npairs, 1) * s.gx * 4 + (size_t)npairs * 4 + nblk_sum) +
      sizeof(double) * std::max(nstate, 1);
  const int P = fit_pairs<T>(ctx, std::max(1, std::min(ctx->batch_pairs_rho, npairs)),
                             std::max(red_bytes, ctx->w_red.bytes + ctx->w_f.bytes) - ctx->w_red.bytes - ctx->w_f.bytes);
  ensure_workspace<T>(ctx, P, K == nullptr);
  upload_f(ctx, f_host, nstate);
  ctx->w_red.ensure(sizeof(double) * ((size_t)std::max(npairs, 1) * s.gx * 4 + (size_t)npairs * 4 + nblk_sum));
  double* red = ctx->w_red.as<double>();
  double* pair_sums = red + (size_t)std::max(npairs, 1) * s.gx * 4;
  if (npairs == 0) LAUNCH(MC_KID_MISC, k_fill, dim3(1024), dim3(256), 0, rho, nnr1, 0.0);
  V* A = ctx->w_a.as<V>();
  const size_t bslab = (size_t)ctx->n3 * ctx->ncols * ctx->n2;
  for (int pair0 = 0; pair0 < npairs; pair0 += P) {
    const int np = std::min(P, npairs - pair0);
    V* B = K ? K + (size_t)pair0 * bslab : ctx->w_b.as<V>();
    with_length(ctx->n3, [&](auto NN) {
      Passes<T, decltype(NN)::value>::zinv(ctx, w, s, np, c0, nstate, pair0, A, red + (size_t)pair0 * s.gx * 4);
    });
    with_length(ctx->n2, [&](auto NN) { Passes<T, decltype(NN)::value>::yinv(ctx, w, s, A, B, np); });
    with_length(ctx->n1, [&](auto NN) {
      Passes<T, decltype(NN)::value>::xrho(ctx, w, s, B, np, pair0, nstate, ctx->w_f.as<double>(), rho, pair0 == 0 ? 1 : 0);
    });
  }
  if (K) {   // the columns of every pair, for the next vpsi on these wavefunctions
    ctx->keep_valid = true;
    ctx->keep_c0 = c0;
    ctx->keep_nstate = nstate;
    ctx->keep_tsize = (int)sizeof(T);
    ctx->keep_epoch = wfn_epoch();
  }
  LAUNCH(MC_KID_MISC, k_rho_sums, dim3(npairs + nblk_sum), dim3(kThreads), 0, red, s.gx, npairs, rho, nnr1, nblk_sum,
         pair_sums);
  std::vector<double> hs((size_t)npairs * 4 + nblk_sum);
  dl_add(ctx, hs.data(), pair_sums, sizeof(double) * hs.size());
  dl_finish(ctx);
  double sg = 0.0, sk = 0.0, sr = 0.0;
  for (int p = 0; p < npairs; ++p) {
    const int is1 = 2 * p, is2 = is1 + 1;
    if (f_host[is1] != 0.0) { sg += f_host[is1] * hs[4 * p + 0]; sk += f_host[is1] * hs[4 * p + 1]; }
    if (is2 < nstate && f_host[is2] != 0.0) { sg += f_host[is2] * hs[4 * p + 2]; sk += f_host[is2] * hs[4 * p + 3]; }
  }
  for (int b = 0; b < nblk_sum; ++b) sr += hs[(size_t)npairs * 4 + b];
  double cr = sr * ctx->omega / ((double)ctx->n1 * ctx->n2 * ctx->n3);
  ctx->last_csumg = sg;
  ctx->last_csumr_raw = cr;
  if (std::is_same<T, float>::value && cr > 0.0 && sg > 0.0) {
    // The FP32 engine contracts norms systematically: its DFT constants and
    // twiddles rounded to FP32 make each 192-point transform scale |x|^2 by
    // 1 - 5.9e-8 on average (the rounded sin(2 pi/3), cos(pi/8), ... lie
    // below their exact values), so the three inverse passes take 1.8e-7 of
    // the charge (csumr - csumg = -1.6e-4 at 1024 electrons).  rho is
    // rescaled so that its integral is the FP64 G-space charge csumg (the
    // invariant of CPMD's csumr / csumg check, rhoofr:625-635); the raw sum
    // stays available through mc_rhoofr_raw_charge.
    const double scale = sg / cr;
    LAUNCH(MC_KID_MISC, k_scale, dim3(1024), dim3(256), 0, rho, nnr1, scale);
    cr *= scale;
  }
  if (ekin) *ekin = sk * ctx->tpiba2;
  if (csumg) *csumg = sg;
  if (csumr) *csumr = cr;
}

// the pass sequence of vpsi over batches of at most P pairs, with the
// workspaces A, B (P pairs each) and the occupations f_dev given
template <typename T>
static void vpsi_run(mc_ctx* ctx, const double2* c0, double2* c2, const double* f_dev, const double* vpot,
                     int nstate, bool acc, int P, v2<T>* A, v2<T>* B, v2<T>* K = nullptr) {
  const WParams w = make_params(ctx);
  const Shapes s = shapes<T>(ctx);
  const int npairs = (nstate + 1) / 2;
  const double scale = 1.0 / ((double)ctx->n1 * ctx->n2 * ctx->n3);
  const size_t bslab = (size_t)ctx->n3 * ctx->ncols * ctx->n2;
  for (int pair0 = 0; pair0 < npairs; pair0 += P) {
    const int np = std::min(P, npairs - pair0);
    if (K) {   // the inverse z and y passes of rhoofr, kept: start from its columns
      B = K + (size_t)pair0 * bslab;
    } else {
      with_length(ctx->n3, [&](auto NN) {
        Passes<T, decltype(NN)::value>::zinv(ctx, w, s, np, c0, nstate, pair0, A, nullptr);
      });
      with_length(ctx->n2, [&](auto NN) { Passes<T, decltype(NN)::value>::yinv(ctx, w, s, A, B, np); });
    }
    with_length(ctx->n1, [&](auto NN) { Passes<T, decltype(NN)::value>::xvpsi(ctx, w, s, B, np, vpot); });
    with_length(ctx->n2, [&](auto NN) { Passes<T, decltype(NN)::value>::yfwd(ctx, w, s, A, B, np); });
    with_length(ctx->n3, [&](auto NN) {
      Passes<T, decltype(NN)::value>::zfwd(ctx, w, s, np, A, c0, c2, f_dev, nstate, pair0, scale, acc ? 1 : 0);
    });
  }
}

template <typename T>
static void vpsi_impl(mc_ctx* ctx, const double2* c0, double2* c2, const double* f_host, const double* vpot,
                      int nstate, bool acc, bool reuse) {
  (void)shapes<T>(ctx);   // rejects unsupported lengths before any allocation
  const int npairs = (nstate + 1) / 2;
  if (npairs == 0) return;
  const size_t f_bytes = sizeof(double) * std::max(nstate, 1);
  WsUse use(ctx->w_a, ctx->w_b);
  // rhoofr's columns of these wavefunctions, if nothing wrote device
  // wavefunctions since (the epoch) and they are still held
  v2<T>* K = nullptr;
  if (reuse && ctx->col_reuse && ctx->keep_valid && ctx->keep_c0 == c0 && ctx->keep_nstate == nstate &&
      ctx->keep_tsize == (int)sizeof(T) && ctx->keep_epoch == wfn_epoch() && ctx->w_keep.p &&
      ctx->w_keep.bytes >= sizeof(v2<T>) * (size_t)npairs * ctx->n3 * ctx->ncols * ctx->n2)
    K = ctx->w_keep.as<v2<T>>();
  ctx->keep_valid = false;   // the x pass below overwrites them
  std::optional<WsUse> use_keep;
  if (K)
    use_keep.emplace(ctx->w_keep, ctx->w_keep);
  else if (mem_limit() != 0)
    ctx->w_keep.release();
  const int P = fit_pairs<T>(ctx, std::max(1, std::min(ctx->batch_pairs_vpsi, npairs)),
                             f_bytes > ctx->w_f.bytes ? f_bytes - ctx->w_f.bytes : 0);
  ensure_workspace<T>(ctx, P, K == nullptr);
  upload_f(ctx, f_host, nstate);
  vpsi_run<T>(ctx, c0, c2, ctx->w_f.as<double>(), vpot, nstate, acc, P, ctx->w_a.as<v2<T>>(),
              K ? nullptr : ctx->w_b.as<v2<T>>(), K);
}

// ---------------------------------------------------------------------------
// Allocation-free vpsi.  The occupations and the transform workspaces live in
// `scratch`, one fixed array per GPU that the code object carries, instead of
// context buffers that grow with hipMalloc.  In host code `scratch` names a
// host-side stand-in: only the address that hipGetSymbolAddress returns for
// the current device (kept per device by scratch_init) is passed to kernels
// and copies.  Every call on one GPU shares the array: calls that overlap in
// time on one GPU (other streams or contexts) race.
// ---------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[MC_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxScratchDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxScratchDevices] = {};

void* scratch_init(int device) {
  MC_CHECK(device >= 0 && device < kMaxScratchDevices, MC_ERR_UNSUPPORTED, "device ordinal beyond 63");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    int cur = -1;
    MC_HIP(hipGetDevice(&cur));
    MC_CHECK(cur == device, MC_ERR_INTERNAL, "scratch_init: device is not current");
    void* p = nullptr;
    MC_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    MC_CHECK(p != nullptr, MC_ERR_HIP, "hipGetSymbolAddress(scratch) returned a null address");
    g_scratch_ptr[device] = p;
  }
  return g_scratch_ptr[device];
}

static size_t round256(size_t b) { return (b + 255) / 256 * 256; }

// the per-kernel timer creates events: it is held off for the call
struct TimerHold {
  mc_ctx* c;
  bool was;
  explicit TimerHold(mc_ctx* ctx) : c(ctx), was(ctx->timer.enabled) { c->timer.enabled = false; }
  ~TimerHold() { c->timer.enabled = was; }
};

template <typename T>
static void vpsi_noalloc_impl(mc_ctx* ctx, const double2* c0, double2* c2, const double* f_host,
                              const double* vpot, int nstate) {
  using V = v2<T>;
  (void)shapes<T>(ctx);
  const int npairs = (nstate + 1) / 2;
  if (npairs == 0) return;
  MC_CHECK(ctx->scratch != nullptr, MC_ERR_INTERNAL, "no scratch address for this device");
  const size_t fbytes = round256(sizeof(double) * (size_t)nstate);
  const size_t abytes = sizeof(V) * (size_t)ctx->n_slots * ctx->n3;           // sticks of one pair
  const size_t bbytes = sizeof(V) * (size_t)ctx->n3 * ctx->ncols * ctx->n2;   // columns of one pair
  const size_t cap = MC_NOALLOC_SCRATCH_BYTES;
  // P pairs take fbytes + round256(P abytes) + P bbytes <= cap
  long long P = 0;
  if (fbytes + 256 < cap) P = (long long)((cap - fbytes - 256) / (abytes + bbytes));
  P = std::min<long long>(P, std::min(ctx->batch_pairs_vpsi, npairs));
  if (P < 1)
    throw Error{MC_ERR_ARG, "mc_vpsi_dev_noalloc: the occupations and one state pair's transform workspaces need " +
                                std::to_string(fbytes + round256(abytes) + bbytes) + " bytes, beyond the " +
                                std::to_string(cap) + "-byte scratch"};
  unsigned char* base = static_cast<unsigned char*>(ctx->scratch);
  double* f_dev = reinterpret_cast<double*>(base);
  V* A = reinterpret_cast<V*>(base + fbytes);
  V* B = reinterpret_cast<V*>(base + fbytes + round256((size_t)P * abytes));
  MC_CHECK(fbytes + round256((size_t)P * abytes) + (size_t)P * bbytes <= cap, MC_ERR_INTERNAL,
           "scratch carving exceeds the array");
  TimerHold hold(ctx);
  MC_HIP(hipMemcpyAsync(f_dev, f_host, sizeof(double) * nstate, hipMemcpyHostToDevice, ctx->stream));
  vpsi_run<T>(ctx, c0, c2, f_dev, vpot, nstate, true, (int)P, A, B);
}

void vpsi_noalloc_dev(mc_ctx* ctx, const double2* c0, double2* c2, const double* f_host, const double* vpot,
                      int nstate) {
  if (ctx->fft_fp32)
    vpsi_noalloc_impl<float>(ctx, c0, c2, f_host, vpot, nstate);
  else
    vpsi_noalloc_impl<double>(ctx, c0, c2, f_host, vpot, nstate);
}

void rhoofr_dev(mc_ctx* ctx, const double2* c0, const double* f_host, int nstate, double* rho, double* ekin,
                double* csumg, double* csumr, bool keep) {
  if (ctx->fft_fp32)
    rhoofr_impl<float>(ctx, c0, f_host, nstate, rho, ekin, csumg, csumr, keep);
  else
    rhoofr_impl<double>(ctx, c0, f_host, nstate, rho, ekin, csumg, csumr, keep);
}

void vpsi_dev(mc_ctx* ctx, const double2* c0, double2* c2, const double* f_host, const double* vpot, int nstate,
              bool acc, bool reuse) {
  if (ctx->fft_fp32)
    vpsi_impl<float>(ctx, c0, c2, f_host, vpot, nstate, acc, reuse);
  else
    vpsi_impl<double>(ctx, c0, c2, f_host, vpot, nstate, acc, reuse);
}

// rows ngw .. ldg-1 of the first n states of c (ld ldg complex rows) <- 0
__global__ void k_zero_pad_rows(double2* __restrict__ c, int ngw, int ldg, int n) {
  const int np = ldg - ngw;
  const size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (t >= (size_t)np * n) return;
  const int col = (int)(t / np), r = ngw + (int)(t - (size_t)col * np);
  c[(size_t)col * ldg + r] = make_double2(0.0, 0.0);
}

void forces_c2_dev(mc_ctx* ctx, const double2* c0, double2* c2, const double* f_host, const double* vpot,
                   int nstate) {
  if (nstate <= 0) return;
  if (ctx->ldg > ctx->ngw) {
    const size_t nt = (size_t)(ctx->ldg - ctx->ngw) * nstate;
    LAUNCH(MC_KID_MISC, k_zero_pad_rows, dim3((unsigned)((nt + 255) / 256)), dim3(256), 0, c2, ctx->ngw, ctx->ldg,
           nstate);
  }
  vpsi_dev(ctx, c0, c2, f_host, vpot, nstate, false, true);
  if (ctx->proj.ready) fnonloc_dev(ctx, c2, f_host, nstate, nullptr);   // no projectors: local potential only
}

}  // namespace mc
