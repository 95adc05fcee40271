// mma.hip -- the method of moving asymptotes (Svanberg) with the design
// vectors in HBM.
//
// Replaces neko-top's mma_t (sources/mma/mma.f90:49-458) and its CPU backend
// (sources/mma/bcknd/cpu/mma_cpu.f90): gensub (:8-184), the dual-primal
// interior-point subsolve (:186-579) and the KKT residual (:581-641).  The
// reference runs all of it on the host; here every n-long operation is a
// fused device stream and only the m-sized quantities (y, lambda, s, mu, z,
// zeta, the (m+1)x(m+1) Newton system) live on the host, which is where the
// reference's MPI_Allreduce calls would hand them over anyway.
//
// Per Newton step the device makes two passes over the n variables:
//   dir  : the search direction's step-length bound
//   eval : the trial point at that step, its residual and the pieces of the
//          Newton system there (repeated while the backtracking line search
//          halves the step; the accepted trial's pieces are the next step's)
// Both are bound by HBM: they read the 9 + 2 m vectors that define the
// subproblem and the iterate, and recompute the direction from them instead
// of storing it (delx, diagx, dx, dxsi, deta and the line search's copies
// were 22 of the 47 vector streams of a step in three passes: newton, dir,
// trial).  At n = 4.2 M, m = 1 dir takes 65 us and eval 84 us (5.7 TB/s)
// where the three passes took 86, 96 and 118 us and each a finalise launch
// and a copy; three updates 40.0 -> 20.4 ms, at n = 20000 (bound by the host
// reads, one per trial) 62 -> 46 ms.  Successive passes run through the
// variables in opposite directions, so a pass begins on what the one before
// left in the 256 MB cache behind the L2s (23.9 ms all in one direction).
// Reductions are deterministic (fixed trees); sums and maxima come back in one
// read per pass.  The reference's default-real literals (0.01, 0.1, 0.9,
// 1.01 in single precision) are kept.  m is a template parameter (1..4).
#include <cmath>
#include <cstring>
#include <vector>

#include "gridsum.h"
#include "internal.h"
#include "nekoamd.h"
#include "reduce.h"

namespace nekoamd {

#define MMA_F0_01 ((double)0.01f)
#define MMA_F0_1 ((double)0.1f)
#define MMA_F0_9 ((double)0.9f)
#define MMA_F1_01 ((double)1.01f)

constexpr int kMmaMaxM = 4;
// Threads per block of an n-pass and most blocks (partials per value): 16
// waves per CU, in few blocks, since each counts itself done at one address;
// the last block has a thread for every partial.
constexpr int kMB = 512;
constexpr int kMG = 512;
constexpr int kMaxVals = 2 + 2 * kMmaMaxM + kMmaMaxM * kMmaMaxM;

struct MmaVec {
  int64_t n;
  double *x, *xsi, *eta, *low, *upp, *alpha, *beta, *xmin, *xmax, *p0j, *q0j;
  double *pij, *qij;  // [i*n + j]
  double *xold1, *xold2;
  double *xt, *xsit, *etat;  // the trial point; swapped with x, xsi, eta
};

struct MmaState {
  int n = 0, m = 0, max_iter = 100;
  double a0 = 0, asyinit = 0.5, asyincr = 1.2, asydecr = 0.7, epsimin = 0;
  double residumax = HUGE_VAL, residunorm = HUGE_VAL, z = 0, zeta = 0;
  std::vector<double> a, c, d, bi, y, lambda, s, mu;
  MmaVec v{};
  double* mem = nullptr;   // one device block for all vectors
  double* part = nullptr;  // kMaxVals * kMG partials
  int* count = nullptr;    // workgroups of the running pass that are done
  bool down = false;       // direction of the update's next pass
  double* bound = nullptr; // the direction pass's result
  // pinned: the last evaluation's results, then the direction pass's
  double* hres = nullptr;
  int newton_iters = 0;    // diagnostics of the last update
};

// ---- reductions ------------------------------------------------------------
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}

// Where a pass's reductions go: block partials, the count of finished
// blocks (0 between passes), and the pinned host memory of the results; dev
// (may be null): the first result for the next pass.
struct MmaOut {
  double* part;
  int* count;
  double* host;
  double* dev;
};

// Reduce K per-thread values over the grid; ismax bit v selects max for
// value v, else sum.  Every block stores its partials past its L2 (device
// scope) and waits for those stores before it counts itself done; the last
// one to do so sums them all, in an order that does not depend on which
// block that is, and writes the results to the host's memory.  That the
// relaxed count cannot be seen before the partials rests on gfx950, not on
// the memory model: a device-scope store has reached memory that all XCDs see
// when vmcnt counts it done, and the barrier keeps thread 0's count behind
// every storing thread's wait.  (A release fence, which the model asks for,
// writes back the whole L2 in every block: 75 us more a pass.)
template <int K>
__device__ __forceinline__ void grid_out(double (&acc)[K], unsigned ismax,
                                         const MmaOut& o) {
  __shared__ double sh[K][kMB / 64];
  __shared__ int last;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int v = 0; v < K; ++v) {
    const double r = (ismax >> v) & 1u ? wave_max(acc[v]) : wave_sum(acc[v]);
    if (lane == 0) sh[v][wv] = r;
  }
  __syncthreads();
  if (threadIdx.x < K) {
    const int v = threadIdx.x;
    double r = sh[v][0];
    for (int q = 1; q < kMB / 64; ++q)
      r = (ismax >> v) & 1u ? fmax(r, sh[v][q]) : r + sh[v][q];
    dev_store(o.part + (int64_t)v * gridDim.x + blockIdx.x, r);
    dev_stores_done();
  }
  __syncthreads();
  if (threadIdx.x == 0)
    last = __hip_atomic_fetch_add(o.count, 1, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT) ==
           (int)gridDim.x - 1;
  __syncthreads();
  if (!last) return;
  static_assert(kMG <= kMB, "one partial per thread");
  const bool in = threadIdx.x < gridDim.x;
  double p[K];
#pragma unroll
  for (int v = 0; v < K; ++v)
    p[v] = in ? dev_load(o.part + (int64_t)v * gridDim.x + threadIdx.x) : 0.0;
#pragma unroll
  for (int v = 0; v < K; ++v) {
    // maxima are of absolute values or at least 1
    const double r = (ismax >> v) & 1u ? wave_max(p[v]) : wave_sum(p[v]);
    if (lane == 0) sh[v][wv] = r;
  }
  __syncthreads();
  if (threadIdx.x < K) {
    const int v = threadIdx.x;
    double r = sh[v][0];
    for (int q = 1; q < kMB / 64; ++q)
      r = (ismax >> v) & 1u ? fmax(r, sh[v][q]) : r + sh[v][q];
    o.host[v] = r;
    if (v == 0 && o.dev != nullptr) *o.dev = r;
  }
  if (threadIdx.x == 0) dev_store(o.count, 0);
}

// ---- per-variable kernels --------------------------------------------------
template <int M>
__global__ void __launch_bounds__(kMB)
    gensub_k(MmaVec V, const double* __restrict__ xd,
             const double* __restrict__ df0dx, const double* __restrict__ dfdx,
             int early, double asyinit, double asyincr, double asydecr,
             MmaOut out) {
  double acc[M];
#pragma unroll
  for (int i = 0; i < M; ++i) acc[i] = 0.0;
  for (int64_t j = (int64_t)blockIdx.x * kMB + threadIdx.x; j < V.n;
       j += (int64_t)gridDim.x * kMB) {
    const double x = xd[j], xmn = V.xmin[j], xmx = V.xmax[j], w = xmx - xmn;
    double lo, up;
    if (early) {
      lo = x - asyinit * w;
      up = x + asyinit * w;
    } else {
      const double x1 = V.xold1[j], x2 = V.xold2[j];
      lo = V.low[j];
      up = V.upp[j];
      const double osc = (x - x1) * (x1 - x2);
      if (osc < 0) {
        lo = x - asydecr * (x1 - lo);
        up = x + asydecr * (up - x1);
      } else if (osc > 0) {
        lo = x - asyincr * (x1 - lo);
        up = x + asyincr * (up - x1);
      } else {
        lo = x - (x1 - lo);
        up = x + (up - x1);
      }
      lo = fmax(lo, x - 10.0 * w);
      lo = fmin(lo, x - MMA_F0_01 * w);
      up = fmin(up, x + 10.0 * w);
      up = fmax(up, x + MMA_F0_01 * w);
    }
    V.low[j] = lo;
    V.upp[j] = up;
    V.alpha[j] = fmax(fmax(xmn, lo + 0.1 * (x - lo)), x - 0.5 * w);
    V.beta[j] = fmin(fmin(xmx, up - MMA_F0_1 * (up - x)), x + 0.5 * w);
    const double reg = 0.00001 / fmax(0.00001, w);
    const double du = (up - x) * (up - x), dl = (x - lo) * (x - lo);
    const double g0 = df0dx[j];
    V.p0j[j] = du * (1.001 * fmax(g0, 0.0) + 0.001 * fmax(-g0, 0.0) + reg);
    V.q0j[j] = dl * (0.001 * fmax(g0, 0.0) + 1.001 * fmax(-g0, 0.0) + reg);
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const double g = dfdx[j * M + i];
      const double p = du * (1.001 * fmax(g, 0.0) + 0.001 * fmax(-g, 0.0) + reg);
      const double q = dl * (0.001 * fmax(g, 0.0) + 1.001 * fmax(-g, 0.0) + reg);
      V.pij[(int64_t)i * V.n + j] = p;
      V.qij[(int64_t)i * V.n + j] = q;
      acc[i] = acc[i] + p / (up - x) + q / (x - lo);
    }
  }
  grid_out<M>(acc, 0u, out);
}

template <int M>
__global__ void __launch_bounds__(kMB) sub_init_k(MmaVec V) {
  for (int64_t j = (int64_t)blockIdx.x * kMB + threadIdx.x; j < V.n;
       j += (int64_t)gridDim.x * kMB) {
    const double x = 0.5 * (V.alpha[j] + V.beta[j]);
    V.x[j] = x;
    V.xsi[j] = fmax(1.0, 1.0 / (x - V.alpha[j]));
    V.eta[j] = fmax(1.0, 1.0 / (V.beta[j] - x));
  }
}

struct Lam {
  double v[kMmaMaxM];
};

// The vectors a pass reads, for variable j.
template <int M>
struct MmaVar {
  double x, xsi, eta, low, upp, alpha, beta, p0, q0, p[M], q[M];
  __device__ __forceinline__ MmaVar(const MmaVec& V, int64_t j)
      : x(V.x[j]), xsi(V.xsi[j]), eta(V.eta[j]), low(V.low[j]), upp(V.upp[j]),
        alpha(V.alpha[j]), beta(V.beta[j]), p0(V.p0j[j]), q0(V.q0j[j]) {
#pragma unroll
    for (int i = 0; i < M; ++i) {
      p[i] = V.pij[(int64_t)i * V.n + j];
      q[i] = V.qij[(int64_t)i * V.n + j];
    }
  }
};

// One variable's part of the Newton system at (x, xsi, eta): the distances
// to the asymptotes and bounds and their reciprocals, the gradients GG_i of
// the constraints, and delx and 1/diagx.
template <int M>
struct MmaNewton {
  double xa, bx, iu, il, ia, ib, GG[M], delx, inv, dpsi;
  __device__ __forceinline__ MmaNewton(const MmaVar<M>& v, double x, double xsi,
                                       double eta, const Lam& lam, double epsi) {
    const double ux = v.upp - x, xl = x - v.low;
    xa = x - v.alpha;
    bx = v.beta - x;
    iu = 1.0 / ux;
    il = 1.0 / xl;
    ia = 1.0 / xa;
    ib = 1.0 / bx;
    const double iu2 = iu * iu, il2 = il * il;
    double pl = 0.0, ql = 0.0;
#pragma unroll
    for (int i = 0; i < M; ++i) {
      pl += v.p[i] * lam.v[i];
      ql += v.q[i] * lam.v[i];
      GG[i] = v.p[i] * iu2 - v.q[i] * il2;
    }
    pl = v.p0 + pl;
    ql = v.q0 + ql;
    dpsi = pl * iu2 - ql * il2;
    delx = dpsi - epsi * ia + epsi * ib;
    inv = 1.0 / (2.0 * (pl * iu2 * iu + ql * il2 * il) + xsi * ia + eta * ib);
  }
};

// The search direction of one variable for the multipliers' dlam.
template <int M>
__device__ __forceinline__ void mma_dir(const MmaNewton<M>& w, double xsi,
                                        double eta, const Lam& dlam,
                                        double epsi, double& dx, double& dxsi,
                                        double& deta) {
  double gl = 0.0;
#pragma unroll
  for (int i = 0; i < M; ++i) gl += w.GG[i] * dlam.v[i];
  dx = -(w.delx + gl) * w.inv;
  dxsi = -xsi + (epsi - dx * xsi) * w.ia;
  deta = -eta + (epsi + dx * eta) * w.ib;
}

// Variable of pass step k of this thread: upwards, or the same ones in the
// opposite order.
__device__ __forceinline__ int64_t pass_var(int64_t n, int64_t k, bool down) {
  const int64_t j = k + (int64_t)blockIdx.x * kMB + threadIdx.x;
  return down ? n - 1 - j : j;
}

// Residual and Newton system pieces at (x, xsi, eta) and lam; with STEP at
// the trial point x + steg dx etc. (the direction of lam, dlam there), which
// it stores, and lam + steg dlam.  bound (may be null): the direction pass's
// result, from which steg is taken as the host takes it (steg then holds the
// bound of the host's own unknowns); so the first trial is queued behind the
// direction pass without a host read between them.
// Values: [sum of rex^2+rexsi^2+reeta^2, max |.|, g_i (M), bb_i (M),
// AA_ik (M*M)].
template <int M, bool STEP>
__global__ void __launch_bounds__(kMB)
    eval_k(MmaVec V, Lam lam, Lam dlam, double epsi, double steg,
           const double* __restrict__ bound, bool down, MmaOut out) {
  constexpr int K = 2 + 2 * M + M * M;
  Lam laml = lam;
  if constexpr (STEP) {
    if (bound != nullptr) steg = 1.0 / fmax(*bound, steg);
#pragma unroll
    for (int i = 0; i < M; ++i)
      laml.v[i] = __dadd_rn(lam.v[i], __dmul_rn(steg, dlam.v[i]));
  }
  double acc[K];
#pragma unroll
  for (int q = 0; q < K; ++q) acc[q] = 0.0;
  for (int64_t k = 0; k < V.n; k += (int64_t)gridDim.x * kMB) {
    const int64_t j = pass_var(V.n, k, down);
    if (j < 0 || j >= V.n) break;
    const MmaVar<M> v(V, j);
    double x = v.x, xsi = v.xsi, eta = v.eta;
    if constexpr (STEP) {
      const MmaNewton<M> o(v, x, xsi, eta, lam, epsi);
      double dx, dxsi, deta;
      mma_dir<M>(o, xsi, eta, dlam, epsi, dx, dxsi, deta);
      x = x + steg * dx;
      xsi = xsi + steg * dxsi;
      eta = eta + steg * deta;
      V.xt[j] = x;
      V.xsit[j] = xsi;
      V.etat[j] = eta;
    }
    const MmaNewton<M> w(v, x, xsi, eta, laml, epsi);
    const double rex = w.dpsi - xsi + eta;
    const double rexsi = xsi * w.xa - epsi;
    const double reeta = eta * w.bx - epsi;
    acc[0] += rex * rex + rexsi * rexsi + reeta * reeta;
    acc[1] = fmax(acc[1], fmax(fabs(rex), fmax(fabs(rexsi), fabs(reeta))));
    const double r = w.delx * w.inv;
#pragma unroll
    for (int i = 0; i < M; ++i) {
      acc[2 + i] += v.p[i] * w.iu + v.q[i] * w.il;
      acc[2 + M + i] += w.GG[i] * r;
#pragma unroll
      for (int q = 0; q < M; ++q)
        acc[2 + 2 * M + i * M + q] += w.GG[i] * w.inv * w.GG[q];
    }
  }
  grid_out<K>(acc, 2u, out);
}

// Value: the search direction's largest step-length bound (max).
template <int M>
__global__ void __launch_bounds__(kMB)
    dir_k(MmaVec V, Lam lam, Lam dlam, double epsi, bool down, MmaOut out) {
  double acc[1] = {1.0};
  for (int64_t k = 0; k < V.n; k += (int64_t)gridDim.x * kMB) {
    const int64_t j = pass_var(V.n, k, down);
    if (j < 0 || j >= V.n) break;
    const MmaVar<M> v(V, j);
    const MmaNewton<M> w(v, v.x, v.xsi, v.eta, lam, epsi);
    double dx, dxsi, deta;
    mma_dir<M>(w, v.xsi, v.eta, dlam, epsi, dx, dxsi, deta);
    double b = fmax(-(MMA_F1_01 * dxsi / v.xsi), -(MMA_F1_01 * deta / v.eta));
    b = fmax(b, -(MMA_F1_01 * dx * w.ia));
    b = fmax(b, MMA_F1_01 * dx * w.ib);
    acc[0] = fmax(acc[0], b);
  }
  grid_out<1>(acc, 1u, out);
}

// KKT pieces at the design x.  Values: [sum of squares, max |.|].
template <int M>
__global__ void __launch_bounds__(kMB)
    kkt_k(MmaVec V, Lam lam, const double* __restrict__ xd,
          const double* __restrict__ df0dx, const double* __restrict__ dfdx,
          MmaOut out) {
  double acc[2] = {0.0, 0.0};
  for (int64_t j = (int64_t)blockIdx.x * kMB + threadIdx.x; j < V.n;
       j += (int64_t)gridDim.x * kMB) {
    double g = 0.0;
#pragma unroll
    for (int i = 0; i < M; ++i) g += dfdx[j * M + i] * lam.v[i];
    const double x = xd[j], xsi = V.xsi[j], eta = V.eta[j];
    const double rex = df0dx[j] + g - xsi + eta;
    const double rexsi = xsi * (x - V.xmin[j]);
    const double reeta = eta * (V.xmax[j] - x);
    acc[0] += rex * rex + rexsi * rexsi + reeta * reeta;
    acc[1] = fmax(acc[1], fmax(fabs(rex), fmax(fabs(rexsi), fabs(reeta))));
  }
  grid_out<2>(acc, 2u, out);
}

// ---- host side -------------------------------------------------------------
static int mma_grid(int64_t n) { return nk_grid(n, kMB, kMG); }

static MmaOut mma_out(MmaState* S) {
  return {S->part, S->count, S->hres, nullptr};
}

// The results of the pass just launched.
static int finish(MmaState* S, int nvals, double* out) {
  NK_LAUNCHED();
  NK_HIP(hipStreamSynchronize(stream()));
  std::memcpy(out, S->hres, sizeof(double) * nvals);
  return kOk;
}

template <int M, bool STEP>
static int evaluate(MmaState* S, int grid, const Lam& lam, const Lam& dlam,
                    double epsi, double steg, const double* bound,
                    double* out) {
  hipLaunchKernelGGL((eval_k<M, STEP>), dim3(grid), dim3(kMB), 0, stream(),
                     S->v, lam, dlam, epsi, steg, bound, S->down, mma_out(S));
  S->down = !S->down;
  return finish(S, 2 + 2 * M + M * M, out);
}

// Gaussian elimination with row partial pivoting (DGESV semantics),
// column-major N x N.  Returns 0 or the 1-based index of a zero pivot.
static int dense_solve(int N, std::vector<double>& A, std::vector<double>& b) {
  int info = 0;
  for (int k = 0; k < N; ++k) {
    int p = k;
    for (int r = k + 1; r < N; ++r)
      if (std::fabs(A[r + k * N]) > std::fabs(A[p + k * N])) p = r;
    if (p != k) {
      for (int c = 0; c < N; ++c) std::swap(A[k + c * N], A[p + c * N]);
      std::swap(b[k], b[p]);
    }
    if (A[k + k * N] == 0.0) {
      if (!info) info = k + 1;
      continue;
    }
    for (int r = k + 1; r < N; ++r) {
      const double l = A[r + k * N] / A[k + k * N];
      A[r + k * N] = l;
      for (int c = k + 1; c < N; ++c) A[r + c * N] -= l * A[k + c * N];
      b[r] -= l * b[k];
    }
  }
  if (info) return info;
  for (int k = N - 1; k >= 0; --k) {
    double s = b[k];
    for (int c = k + 1; c < N; ++c) s -= A[k + c * N] * b[c];
    b[k] = s / A[k + k * N];
  }
  return 0;
}

struct Small {
  double max = 0.0, sq = 0.0;
};

// The m-sized residuals (rey, rez, relambda, remu, rezeta, res).
static Small small_resid(const MmaState* S, const double* g, const double* y,
                         double z, const double* lam, const double* mu,
                         double zeta, const double* s, double epsi) {
  Small r;
  double la = 0.0;
  for (int i = 0; i < S->m; ++i) la += lam[i] * S->a[i];
  const double rez = S->a0 - zeta - la, rezeta = zeta * z - epsi;
  for (int i = 0; i < S->m; ++i) {
    const double rey = S->c[i] + S->d[i] * y[i] - lam[i] - mu[i];
    const double rel = g[i] - S->a[i] * z - y[i] + s[i] - S->bi[i];
    const double remu = mu[i] * y[i] - epsi;
    const double res = lam[i] * s[i] - epsi;
    r.max = std::fmax(r.max, std::fmax(std::fmax(std::fabs(rey), std::fabs(rel)),
                                       std::fmax(std::fabs(remu), std::fabs(res))));
    r.sq += rey * rey + rel * rel + remu * remu + res * res;
  }
  r.max = std::fmax(r.max, std::fmax(std::fabs(rez), std::fabs(rezeta)));
  r.sq += rez * rez + rezeta * rezeta;
  return r;
}

template <int M>
static int mma_update_t(MmaState* S, int iter, double* xd, const double* df0dx,
                        const double* fval, const double* dfdx) {
  MmaVec& V = S->v;
  const int grid = mma_grid(V.n);
  double out[kMaxVals];
  // the order of an update's sums must not depend on the updates before it
  S->down = false;
  // ---- gensub
  hipLaunchKernelGGL((gensub_k<M>), dim3(grid), dim3(kMB), 0, stream(), V, xd,
                     df0dx, dfdx, iter < 3 ? 1 : 0, S->asyinit, S->asyincr,
                     S->asydecr, mma_out(S));
  int rc = finish(S, M, out);
  if (rc) return rc;
  for (int i = 0; i < M; ++i) S->bi[i] = out[i] - fval[i];
  // ---- subsolve
  double epsi = 1.0, z = 1.0, zeta = 1.0;
  double y[M], lam[M], s[M], mu[M];
  for (int i = 0; i < M; ++i) {
    y[i] = 1.0;
    lam[i] = 1.0;
    s[i] = 1.0;
    mu[i] = std::fmax(1.0, 0.5 * S->c[i]);
  }
  hipLaunchKernelGGL((sub_init_k<M>), dim3(grid), dim3(kMB), 0, stream(), V);
  NK_LAUNCHED();
  S->newton_iters = 0;
  while (epsi > MMA_F0_9 * S->epsimin) {
    Lam L{};
    for (int i = 0; i < M; ++i) L.v[i] = lam[i];
    rc = evaluate<M, false>(S, grid, L, L, epsi, 0.0, nullptr, out);
    if (rc) return rc;
    Small sm = small_resid(S, out + 2, y, z, lam, mu, zeta, s, epsi);
    double residumax = std::fmax(out[1], sm.max);
    double residunorm = std::sqrt(sm.sq + out[0]);
    for (int it = 1; it <= S->max_iter; ++it) {
      if (residumax < epsi) break;
      ++S->newton_iters;
      for (int i = 0; i < M; ++i) L.v[i] = lam[i];
      // the pieces of the last evaluation, which was at this point
      const double* g = out + 2;
      const double* bbs = out + 2 + M;
      const double* AAs = out + 2 + 2 * M;
      double la = 0.0;
      for (int i = 0; i < M; ++i) la += lam[i] * S->a[i];
      const double delz = S->a0 - la - epsi / z;
      double dely[M];
      std::vector<double> A((M + 1) * (M + 1), 0.0), bb(M + 1, 0.0);
      for (int i = 0; i < M; ++i) {
        dely[i] = S->c[i] + S->d[i] * y[i] - lam[i] - epsi / y[i];
        const double dellam = g[i] - S->a[i] * z - y[i] - S->bi[i] + epsi / lam[i];
        bb[i] = dellam + dely[i] / (S->d[i] + mu[i] / y[i]) - bbs[i];
      }
      bb[M] = delz;
      for (int i = 0; i < M; ++i)
        for (int k = 0; k < M; ++k) A[i + k * (M + 1)] = AAs[i * M + k];
      for (int i = 0; i < M; ++i) {
        A[i + i * (M + 1)] += s[i] / lam[i] + 1.0 / (S->d[i] + mu[i] / y[i]);
        A[i + M * (M + 1)] = S->a[i];
        A[M + i * (M + 1)] = S->a[i];
      }
      A[M + M * (M + 1)] = -zeta / z;
      const int info = dense_solve(M + 1, A, bb);
      if (info) {
        set_error("mma_update", "the (m+1) Newton system is singular (DGESV)");
        return kErrNumeric;
      }
      double dlam[M], dy[M], dmu[M], ds[M];
      for (int i = 0; i < M; ++i) dlam[i] = bb[i];
      const double dz = bb[M];
      for (int i = 0; i < M; ++i) {
        dy[i] = (-dely[i] + dlam[i]) / (S->d[i] + mu[i] / y[i]);
        dmu[i] = -mu[i] + (epsi - mu[i] * dy[i]) / y[i];
        ds[i] = -s[i] + (epsi - dlam[i] * s[i]) / lam[i];
      }
      const double dzeta = -zeta + (epsi - zeta * dz) / z;
      Lam DL{};
      for (int i = 0; i < M; ++i) DL.v[i] = dlam[i];
      MmaOut dout = mma_out(S);
      dout.host = S->hres + kMaxVals;
      dout.dev = S->bound;
      hipLaunchKernelGGL((dir_k<M>), dim3(grid), dim3(kMB), 0, stream(), V, L,
                         DL, epsi, S->down, dout);
      S->down = !S->down;
      NK_LAUNCHED();
      double steg = 1.0;
      for (int i = 0; i < M; ++i) {
        steg = std::fmax(steg, -(MMA_F1_01 * dy[i] / y[i]));
        steg = std::fmax(steg, -(MMA_F1_01 * dlam[i] / lam[i]));
        steg = std::fmax(steg, -(MMA_F1_01 * dmu[i] / mu[i]));
        steg = std::fmax(steg, -(MMA_F1_01 * ds[i] / s[i]));
      }
      steg = std::fmax(steg, -(MMA_F1_01 * dz / z));
      steg = std::fmax(steg, -(MMA_F1_01 * dzeta / zeta));
      double yo[M], lo[M], so[M], muo[M];
      std::memcpy(yo, y, sizeof(y));
      std::memcpy(lo, lam, sizeof(lam));
      std::memcpy(so, s, sizeof(s));
      std::memcpy(muo, mu, sizeof(mu));
      const double zo = z, zetao = zeta;
      double newresidu = 2.0 * residunorm, newmax = residumax;
      int itto = 0;
      while (newresidu > residunorm && itto < 50) {
        ++itto;
        rc = evaluate<M, true>(S, grid, L, DL, epsi, steg,
                               itto == 1 ? S->bound : nullptr, out);
        if (rc) return rc;
        if (itto == 1) steg = 1.0 / std::fmax(S->hres[kMaxVals], steg);
        for (int i = 0; i < M; ++i) {
          y[i] = yo[i] + steg * dy[i];
          lam[i] = lo[i] + steg * dlam[i];
          mu[i] = muo[i] + steg * dmu[i];
          s[i] = so[i] + steg * ds[i];
        }
        z = zo + steg * dz;
        zeta = zetao + steg * dzeta;
        sm = small_resid(S, out + 2, y, z, lam, mu, zeta, s, epsi);
        newresidu = std::sqrt(sm.sq + out[0]);
        newmax = std::fmax(out[1], sm.max);
        steg = steg / 2.0;
      }
      // the last trial is the new point; there is none if the residual to
      // improve on is not finite
      if (itto > 0) {
        std::swap(V.x, V.xt);
        std::swap(V.xsi, V.xsit);
        std::swap(V.eta, V.etat);
      }
      residunorm = newresidu;
      residumax = newmax;
    }
    epsi = 0.1 * epsi;
  }
  // xold2 <- xold1 <- design x ; design x <- x
  NK_HIP(hipMemcpyAsync(V.xold2, V.xold1, sizeof(double) * V.n,
                        hipMemcpyDeviceToDevice, stream()));
  NK_HIP(hipMemcpyAsync(V.xold1, xd, sizeof(double) * V.n,
                        hipMemcpyDeviceToDevice, stream()));
  NK_HIP(hipMemcpyAsync(xd, V.x, sizeof(double) * V.n,
                        hipMemcpyDeviceToDevice, stream()));
  for (int i = 0; i < M; ++i) {
    S->y[i] = y[i];
    S->lambda[i] = lam[i];
    S->s[i] = s[i];
    S->mu[i] = mu[i];
  }
  S->z = z;
  S->zeta = zeta;
  NK_HIP(hipStreamSynchronize(stream()));
  return kOk;
}

template <int M>
static int mma_kkt_t(MmaState* S, const double* xd, const double* df0dx,
                     const double* fval, const double* dfdx) {
  const int grid = mma_grid(S->v.n);
  Lam L{};
  for (int i = 0; i < M; ++i) L.v[i] = S->lambda[i];
  hipLaunchKernelGGL((kkt_k<M>), dim3(grid), dim3(kMB), 0, stream(), S->v, L,
                     xd, df0dx, dfdx, mma_out(S));
  double out[2];
  int rc = finish(S, 2, out);
  if (rc) return rc;
  double mx = out[1], sq = 0.0, la = 0.0;
  for (int i = 0; i < M; ++i) la += S->lambda[i] * S->a[i];
  const double rez = S->a0 - S->zeta - la, rezeta = S->zeta * S->z;
  for (int i = 0; i < M; ++i) {
    const double rey = S->c[i] + S->d[i] * S->y[i] - S->lambda[i] - S->mu[i];
    const double rel = fval[i] - S->a[i] * S->z - S->y[i] + S->s[i];
    const double remu = S->mu[i] * S->y[i], res = S->lambda[i] * S->s[i];
    mx = std::fmax(mx, std::fmax(std::fmax(std::fabs(rey), std::fabs(rel)),
                                 std::fmax(std::fabs(remu), std::fabs(res))));
    sq += rey * rey + rel * rel + remu * remu + res * res;
  }
  mx = std::fmax(mx, std::fmax(std::fabs(rez), std::fabs(rezeta)));
  sq += rez * rez + rezeta * rezeta;
  S->residumax = mx;
  S->residunorm = std::sqrt(sq + out[0]);
  return kOk;
}

}  // namespace nekoamd

using namespace nekoamd;

extern "C" {

int nekoamd_mma_create(void** mma, const int* n, const int* m, const void* x,
                       const double* a0, const double* a, const double* c,
                       const double* d, const void* xmin, const void* xmax,
                       const int* max_iter, const double* epsimin,
                       const double* asyinit, const double* asyincr,
                       const double* asydecr) {
  NK_INIT();
  NK_REQUIRE(mma && n && m && x && a0 && a && c && d && xmin && xmax &&
                 max_iter && epsimin && asyinit && asyincr && asydecr,
             "null argument");
  NK_REQUIRE(*n > 0, "n must be positive");
  NK_REQUIRE(*m >= 1 && *m <= kMmaMaxM, "m must be in [1, 4]");
  MmaState* S = new MmaState();
  S->n = *n;
  S->m = *m;
  S->max_iter = *max_iter;
  S->a0 = *a0;
  S->asyinit = *asyinit;
  S->asyincr = *asyincr;
  S->asydecr = *asydecr;
  S->epsimin = *epsimin > 0 ? *epsimin : 1.0e-9 * std::sqrt((double)(*m + *n));
  S->a.assign(a, a + *m);
  S->c.assign(c, c + *m);
  S->d.assign(d, d + *m);
  S->bi.assign(*m, 0.0);
  S->y.assign(*m, 0.0);
  S->lambda.assign(*m, 0.0);
  S->s.assign(*m, 0.0);
  S->mu.assign(*m, 0.0);
  const int64_t N = *n;
  const size_t nvec = 16 + 2 * (size_t)*m;
  hipError_t e = hipMalloc((void**)&S->mem, sizeof(double) * nvec * N);
  if (e == hipSuccess)
    e = hipMalloc((void**)&S->part, sizeof(double) * kMaxVals * kMG);
  if (e == hipSuccess) e = hipMalloc((void**)&S->count, sizeof(int));
  if (e == hipSuccess) e = hipMemset(S->count, 0, sizeof(int));
  if (e == hipSuccess) e = hipMalloc((void**)&S->bound, sizeof(double));
  if (e == hipSuccess)
    e = hipHostMalloc((void**)&S->hres, sizeof(double) * (kMaxVals + 1),
                      hipHostMallocDefault);
  if (e != hipSuccess) {
    if (S->mem) (void)hipFree(S->mem);
    if (S->part) (void)hipFree(S->part);
    if (S->count) (void)hipFree(S->count);
    if (S->bound) (void)hipFree(S->bound);
    delete S;
    return fail_hip(__func__, e);
  }
  double* p = S->mem;
  MmaVec& V = S->v;
  V.n = N;
  double** slots[] = {&V.x,     &V.xsi,   &V.eta,   &V.low,    &V.upp,
                      &V.alpha, &V.beta,  &V.xmin,  &V.xmax,   &V.p0j,
                      &V.q0j,   &V.xold1, &V.xold2, &V.xt,     &V.xsit,
                      &V.etat};
  for (double** s : slots) {
    *s = p;
    p += N;
  }
  V.pij = p;
  p += (size_t)*m * N;
  V.qij = p;
  // initial state (mma.f90:132-184): xold1 = xold2 = x, low = min x, upp = max x
  std::vector<double> hx(N);
  e = hipMemcpy(hx.data(), x, sizeof(double) * N, hipMemcpyDeviceToHost);
  if (e == hipSuccess)
    e = hipMemcpy(V.xold1, x, sizeof(double) * N, hipMemcpyDeviceToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(V.xold2, x, sizeof(double) * N, hipMemcpyDeviceToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(V.xmin, xmin, sizeof(double) * N, hipMemcpyDeviceToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(V.xmax, xmax, sizeof(double) * N, hipMemcpyDeviceToDevice);
  if (e != hipSuccess) {
    (void)hipFree(S->mem);
    (void)hipFree(S->part);
    (void)hipFree(S->count);
    (void)hipFree(S->bound);
    (void)hipHostFree(S->hres);
    delete S;
    return fail_hip(__func__, e);
  }
  double lo = hx[0], hi = hx[0];
  for (int64_t j = 1; j < N; ++j) {
    lo = std::fmin(lo, hx[j]);
    hi = std::fmax(hi, hx[j]);
  }
  int rc = nekoamd_cfill(V.low, &lo, &V.n);
  if (!rc) rc = nekoamd_cfill(V.upp, &hi, &V.n);
  if (rc) {
    (void)hipFree(S->mem);
    (void)hipFree(S->part);
    (void)hipFree(S->count);
    (void)hipFree(S->bound);
    (void)hipHostFree(S->hres);
    delete S;
    return rc;
  }
  *mma = S;
  return kOk;
}

int nekoamd_mma_free(void* mma) {
  MmaState* S = (MmaState*)mma;
  if (!S) return kOk;
  NK_HIP(hipStreamSynchronize(stream()));
  if (S->mem) NK_HIP(hipFree(S->mem));
  if (S->part) NK_HIP(hipFree(S->part));
  if (S->count) NK_HIP(hipFree(S->count));
  if (S->bound) NK_HIP(hipFree(S->bound));
  if (S->hres) NK_HIP(hipHostFree(S->hres));
  delete S;
  return kOk;
}

// x (device, n) is replaced by the new design; dfdx is m x n column-major
// on the device (the reference's dfdx(m, n)); fval on the host (m).
int nekoamd_mma_update(void* mma, const int* iter, void* x, const void* df0dx,
                       const double* fval, const void* dfdx) {
  NK_INIT();
  MmaState* S = (MmaState*)mma;
  NK_REQUIRE(S && iter && x && df0dx && fval && dfdx, "null argument");
  switch (S->m) {
    case 1: return mma_update_t<1>(S, *iter, (double*)x, (const double*)df0dx, fval, (const double*)dfdx);
    case 2: return mma_update_t<2>(S, *iter, (double*)x, (const double*)df0dx, fval, (const double*)dfdx);
    case 3: return mma_update_t<3>(S, *iter, (double*)x, (const double*)df0dx, fval, (const double*)dfdx);
    default: return mma_update_t<4>(S, *iter, (double*)x, (const double*)df0dx, fval, (const double*)dfdx);
  }
}

int nekoamd_mma_kkt(void* mma, const void* x, const void* df0dx,
                    const double* fval, const void* dfdx) {
  NK_INIT();
  MmaState* S = (MmaState*)mma;
  NK_REQUIRE(S && x && df0dx && fval && dfdx, "null argument");
  switch (S->m) {
    case 1: return mma_kkt_t<1>(S, (const double*)x, (const double*)df0dx, fval, (const double*)dfdx);
    case 2: return mma_kkt_t<2>(S, (const double*)x, (const double*)df0dx, fval, (const double*)dfdx);
    case 3: return mma_kkt_t<3>(S, (const double*)x, (const double*)df0dx, fval, (const double*)dfdx);
    default: return mma_kkt_t<4>(S, (const double*)x, (const double*)df0dx, fval, (const double*)dfdx);
  }
}

// res[0] = residumax, res[1] = residunorm, res[2] = Newton iterations of
// the last update.
int nekoamd_mma_residuals(void* mma, double* res) {
  MmaState* S = (MmaState*)mma;
  NK_REQUIRE(S && res, "null argument");
  res[0] = S->residumax;
  res[1] = S->residunorm;
  res[2] = S->newton_iters;
  return kOk;
}

// Host copies of the m-sized duals: y, lambda, s, mu (m each), zs = {z, zeta}.
int nekoamd_mma_duals(void* mma, double* y, double* lambda, double* s,
                      double* mu, double* zs) {
  MmaState* S = (MmaState*)mma;
  NK_REQUIRE(S && y && lambda && s && mu && zs, "null argument");
  for (int i = 0; i < S->m; ++i) {
    y[i] = S->y[i];
    lambda[i] = S->lambda[i];
    s[i] = S->s[i];
    mu[i] = S->mu[i];
  }
  zs[0] = S->z;
  zs[1] = S->zeta;
  return kOk;
}

}  // extern "C"
