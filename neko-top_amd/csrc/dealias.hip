// dealias.hip -- dealiased (over-integrated) advection: the velocity fields
// are interpolated from the lx GLL points to lxd = 3 lx / 2 Gauss-Legendre
// (GL) points per direction, the convective products are formed and
// weighted there, and the result returns to GLL through the transpose of the
// interpolation (a weak-form projection).  The three operators of
// sources/adjoint/adv_adjoint_dealias.f90 and Neko's dealiased forward term:
//
//   forward    f_c = beta f_c - J^T [ t . opgrad(t_c) ]               (Neko
//              adv_dealias_t%compute)
//   linearised f_c = beta f_c - J^T [ u' . opgrad(U_c) + U . opgrad(u'_c) ]
//              (compute_linear_advection_dealias :466-653)
//   adjoint    f_c = beta f_c - J^T [ sum_d a_d opgrad_c(U_d)
//                                     + sum_b D_b^T (w3 a_c sum_d U_d c_b[d]) ]
//              (compute_adjoint_advection_dealias :227-449)
//
// with t = (J x J x J) u on the GL points, opgrad_a(f) = w3 sum_b c_b[a]
// d_b f, w3 the GL tensor weights and c_b[a] the GL metric: the GLL cofactors
// interpolated to GL, as init_dealias builds coef_GL (:155-163).
//
// One workgroup per element does everything on chip: the GLL rows are read
// straight into registers, interpolated to GL by three in-place tensor
// passes, combined point by point, and mapped back by three transposed
// passes straight into f.  The reference's device branch makes ~20 round
// trips through n_GL-sized HBM arrays per call; here HBM sees the GLL inputs,
// the GL metric and f once (174 KB per element for the adjoint at lx = 8,
// 0.8 ms at 32^3; its 1.5 MFLOP take 0.6 ms at the FP64 rate).
//
// Measured at 32^3 p=7, before (two LDS reads per FMA) and now (one line per
// thread, see dealias_k): forward 4.03 -> 1.24 ms, linearised 7.24 -> 2.24,
// adjoint 6.98 -> 1.76; 13x11x9 p=5 forward 43.2 -> 22.3 us.
#include <cmath>
#include <vector>

#include "internal.h"
#include "nekoamd.h"
#include "uniform.h"

namespace nekoamd {
namespace {

constexpr int kFwd = 0, kLin = 1, kAdj = 2;

template <int LXD>
constexpr int dl_threads() {
  return LXD == 12 ? 512 : 256;
}

struct DealiasState {
  int lx = 0, lxd = 0, nelv = 0;
  int64_t n = 0, ngl = 0;
  double* cof = nullptr;   // [9][ngl], row m = 3b + a holds c_b[a]
  // J [lxd*lx] | Dg [lxd*lxd] | wg [lxd] | J^T [lx*lxd] | Dg^T [lxd*lxd]
  double* mats = nullptr;
};

// LDS of one element: the 1-D matrices, the two interpolation temporaries
// (t2 also stages one GLL input field) and NB GL-point fields.
template <int LX, int LXD, int NB>
struct DlShared {
  double J[LXD * LX];
  double Dg[LXD * LXD];
  double w[LXD];
  double t1[LXD * LX * LX];
  double t2[LXD * LXD * LX];
  double buf[NB][LXD * LXD * LXD];
};

template <int LX, int LXD, int NB>
__device__ __forceinline__ void load_mats(DlShared<LX, LXD, NB>& sh,
                                          const double* __restrict__ mats) {
  constexpr int NT = dl_threads<LXD>();
  for (int i = threadIdx.x; i < LXD * LX; i += NT) sh.J[i] = mats[i];
  for (int i = threadIdx.x; i < LXD * LXD; i += NT)
    sh.Dg[i] = mats[LXD * LX + i];
  for (int i = threadIdx.x; i < LXD; i += NT)
    sh.w[i] = mats[LXD * LX + LXD * LXD + i];
}

// dst (GL, LDS) = (J x J x J) sh.t2[0 .. LX^3), the staged GLL field.  The
// caller synchronised after staging; returns synchronised.
template <int LX, int LXD, int NB>
__device__ __forceinline__ void interp_up(DlShared<LX, LXD, NB>& sh,
                                          double* dst) {
  constexpr int NT = dl_threads<LXD>();
  constexpr int NPG = LXD * LXD * LXD;
  for (int p = threadIdx.x; p < LXD * LX * LX; p += NT) {
    const int q = p % LXD, jk = p / LXD;
    double s = 0.0;
#pragma unroll
    for (int l = 0; l < LX; ++l) s += sh.J[q * LX + l] * sh.t2[l + LX * jk];
    sh.t1[p] = s;
  }
  __syncthreads();
  for (int p = threadIdx.x; p < LXD * LXD * LX; p += NT) {
    const int q = p % LXD, r = (p / LXD) % LXD, k = p / (LXD * LXD);
    double s = 0.0;
#pragma unroll
    for (int l = 0; l < LX; ++l)
      s += sh.J[r * LX + l] * sh.t1[q + LXD * (l + LX * k)];
    sh.t2[p] = s;
  }
  __syncthreads();
  for (int p = threadIdx.x; p < NPG; p += NT) {
    const int qr = p % (LXD * LXD), tt = p / (LXD * LXD);
    double s = 0.0;
#pragma unroll
    for (int l = 0; l < LX; ++l)
      s += sh.J[tt * LX + l] * sh.t2[qr + LXD * LXD * l];
    dst[p] = s;
  }
  __syncthreads();
}

// ---- the operators -------------------------------------------------------

// LDS layout of a GL-sized field: row stride RS and plane stride PS in
// doubles.  An even lxd gets one double of padding per row, so that the 64
// lanes of a wave that read along r (stride RS) fall on distinct banks (at
// lxd = 12 a stride of 12 doubles would use a quarter of them).
template <int LX, int LXD>
struct Dl {
  static constexpr int NL = LXD * LXD;        // lines of one direction
  static constexpr int NO = 3 * NL;           // working threads
  static constexpr int NT = (NO + 63) / 64 * 64;
  static constexpr int PPT = LXD / 3;         // points per thread
  static constexpr int NP = LX * LX * LX, NPG = NL * LXD;
  static constexpr int RS = LXD % 2 ? LXD : LXD + 1;
  static constexpr int PS = RS * LXD;
  static constexpr int BUF = PS * LXD;
  static_assert(LXD == 3 * LX / 2 && LXD % 3 == 0, "points per thread");
  static_assert(6 * LX * LX <= NT, "one thread per GLL row of six fields");
};

// Offsets of the 1-D operators in `mats`.
template <int LX, int LXD>
struct DlMats {
  static constexpr int J = 0, Dg = LXD * LX, w = Dg + LXD * LXD, JT = w + LXD,
                       DgT = JT + LX * LXD, size = DgT + LXD * LXD;
};

// out[q] = sum_l M[q NI + l] in[l], l in order.  M is one of the 1-D
// operators, the same for every lane, so its rows come by scalar loads and
// enter the FMAs as scalar operands.  A row is requested once the first
// product of the row before it is formed: two rows are in flight at most.
template <int NI, int NQ>
__device__ __forceinline__ void dl_apply(const double* __restrict__ M,
                                         const double (&in)[NI],
                                         double (&out)[NQ]) {
  double row[NI], next[NI];
  {
    const auto m = uniform_row(M, in[0]);
#pragma unroll
    for (int l = 0; l < NI; ++l) row[l] = m[l];
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    double s = row[0] * in[0];
    if (q + 1 < NQ) {
      const auto m = uniform_row(M + (q + 1) * NI, s);
#pragma unroll
      for (int l = 0; l < NI; ++l) next[l] = m[l];
    }
#pragma unroll
    for (int l = 1; l < NI; ++l) s += row[l] * in[l];
    out[q] = s;
    if (q + 1 < NQ) {
#pragma unroll
      for (int l = 0; l < NI; ++l) row[l] = next[l];
    }
  }
}

// One line of a tensor pass in place: NI values at p[l str] become NQ values
// at p[q str].
template <int NI, int NQ>
__device__ __forceinline__ void dl_line(const double* __restrict__ M, double* p,
                                        int str) {
  double in[NI], out[NQ];
#pragma unroll
  for (int l = 0; l < NI; ++l) in[l] = p[l * str];
  dl_apply<NI, NQ>(M, in, out);
#pragma unroll
  for (int q = 0; q < NQ; ++q) p[q * str] = out[q];
}

// Line t of the 3 NL lines of a GL field (NL along r, then s, then t):
// its first value's offset and its stride.
template <int LX, int LXD>
__device__ __forceinline__ void dl_dir_line(int t, int& base, int& str) {
  using S = Dl<LX, LXD>;
  const int b = t / S::NL, l = t % S::NL, lo = l % LXD, hi = l / LXD;
  base = b == 0 ? S::RS * lo + S::PS * hi : b == 1 ? lo + S::PS * hi : lo + S::RS * hi;
  str = b == 0 ? 1 : b == 1 ? S::RS : S::PS;
}

// Three fields (J x J x J)-interpolated into bf: thread t in [t0, t0 + 3 lx^2)
// holds GLL row t - t0 in g.  Returns synchronised.
template <int LX, int LXD>
__device__ __forceinline__ void dl_up(double* bf,
                                      const double* __restrict__ mats,
                                      const double (&g)[LX], int t0) {
  using S = Dl<LX, LXD>;
  const double* J = mats + DlMats<LX, LXD>::J;
  const int t = threadIdx.x, tr = t - t0;
  if (tr >= 0 && tr < 3 * LX * LX) {
    const int f = tr / (LX * LX), l = tr % (LX * LX);
    double* p = bf + f * S::BUF + S::RS * (l % LX) + S::PS * (l / LX);
    double out[LXD];
    dl_apply<LX, LXD>(J, g, out);
#pragma unroll
    for (int q = 0; q < LXD; ++q) p[q] = out[q];
  }
  __syncthreads();
  if (t < 3 * LXD * LX) {
    const int f = t / (LXD * LX), l = t % (LXD * LX);
    dl_line<LX, LXD>(J, bf + f * S::BUF + l % LXD + S::PS * (l / LXD), S::RS);
  }
  __syncthreads();
  if (t < S::NO) {
    const int f = t / S::NL, l = t % S::NL;
    dl_line<LX, LXD>(J, bf + f * S::BUF + l % LXD + S::RS * (l / LXD), S::PS);
  }
  __syncthreads();
}

template <int LX>
__device__ __forceinline__ void dl_row(double (&g)[LX],
                                       const double* __restrict__ a0,
                                       const double* __restrict__ a1,
                                       const double* __restrict__ a2,
                                       int64_t eb, int r) {
  const int f = r / (LX * LX);
  const double* a = (f == 0 ? a0 : f == 1 ? a1 : a2) + eb + (int64_t)LX * (r % (LX * LX));
#pragma unroll
  for (int l = 0; l < LX; ++l) g[l] = a[l];
}

constexpr int kDlFields = 5;  // GL-sized LDS fields: b[3] and x[2]

// a*: forward u,v,w; linearised u'; adjoint the adjoint velocity.
// b*: the base flow U (linearised and adjoint).
//
// Every tensor pass is a set of lines: a thread reads the line's values once
// from LDS, forms all of the line's outputs with the 1-D operator in scalar
// registers and writes them back, so a pass costs one LDS read and one write
// per value (the first form of this kernel read two LDS values per FMA and
// was bound by them).  The three directions of a gradient are 3 lxd^2 lines
// of one pass (432 threads at lxd = 12); between passes the same threads own
// lxd / 3 points each, whose pointwise factors stay in registers:
//
//   forward  O_c = sum_b C_b d_b t_c,       C_b = w3 sum_a c_b[a] t_a
//   linear   O_c = sum_b C'_b d_b U_c + C_b d_b u'_c
//   adjoint  O_c = w3 sum_b c_b[c] E_b + sum_b D_b^T (a_c C_b),
//            E_b = sum_d a_d d_b U_d,       C_b = w3 sum_d c_b[d] U_d
//
// (contravariant components: the metric is read once per point, and
// opgrad_c(U_d) is never formed).  Five GL fields of LDS (75 KB at lxd = 12)
// leave room for two elements per CU; interpolation and map-back run in
// place in them.  The linearised operator needs both sets' C_b and is held
// to 128 registers so that two workgroups fit (2.24 ms with 16 spilled
// registers against 2.82 ms without the cap at 32^3 p=7).
template <int LX, int LXD, int MODE>
__global__ void __launch_bounds__((Dl<LX, LXD>::NT), (MODE == kLin ? 4 : 1))
    dealias_k(double* __restrict__ fx, double* __restrict__ fy,
              double* __restrict__ fz, const double* __restrict__ a0,
              const double* __restrict__ a1, const double* __restrict__ a2,
              const double* __restrict__ b0, const double* __restrict__ b1,
              const double* __restrict__ b2, const double* __restrict__ cof,
              const double* __restrict__ mats, int64_t ngl, double beta) {
  using S = Dl<LX, LXD>;
  using M = DlMats<LX, LXD>;
  constexpr int PPT = S::PPT, NO = S::NO, R3 = 3 * LX * LX;
  __shared__ double sh[kDlFields][S::BUF];
  double (*const B)[S::BUF] = sh;
  double (*const X)[S::BUF] = sh + 3;
  const int t = threadIdx.x;
  const bool on = t < NO;
  const int64_t eb = (int64_t)blockIdx.x * S::NP, gb = (int64_t)blockIdx.x * S::NPG;

  // GLL rows of the fields, all requested before the first pass
  double g[LX];
  if constexpr (MODE == kFwd) {
    if (t < R3) dl_row<LX>(g, a0, a1, a2, eb, t);
  } else {
    if (t < R3)
      dl_row<LX>(g, a0, a1, a2, eb, t);
    else if (t < 2 * R3)
      dl_row<LX>(g, b0, b1, b2, eb, t - R3);
  }

  // the thread's points p = t + q NO: (i, j) the same for all of them,
  // k = t / NL + 3 q
  const int ij = t % S::NL, i = ij % LXD, j = ij / LXD, k0 = t / S::NL;
  const int at0 = i + S::RS * j + S::PS * k0;  // + 3 PS q
  const double* w = mats + M::w;
  const double wij = on ? w[i] * w[j] : 0.0;
  int lb = 0, ls = 0;
  if (on) dl_dir_line<LX, LXD>(t, lb, ls);
  const int db = on ? t / S::NL : 0;  // the line's direction

  double O[3][PPT];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int q = 0; q < PPT; ++q) O[c][q] = 0.0;

  // C_b at point q from three fields' values there
  auto metric = [&](int q, double (&c9)[9]) {
    const int64_t p = gb + t + q * NO;
#pragma unroll
    for (int m = 0; m < 9; ++m)
      c9[m] = __builtin_nontemporal_load(cof + m * ngl + p);
  };
  // O_c += sum_b C_b d_b (field c of B); B is consumed
  auto convect = [&](const double (&Cb)[3][PPT]) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double in[LXD], out[LXD];
      if (on) {
#pragma unroll
        for (int l = 0; l < LXD; ++l) in[l] = B[c][lb + l * ls];
        dl_apply<LXD, LXD>(mats + M::Dg, in, out);
      }
      __syncthreads();  // rows of field c and the sums of field c - 1 read
      if (on) {
        double* o = db == 0 ? X[0] : db == 1 ? X[1] : B[c];
#pragma unroll
        for (int l = 0; l < LXD; ++l) o[lb + l * ls] = out[l];
      }
      __syncthreads();
      if (on) {
#pragma unroll
        for (int q = 0; q < PPT; ++q) {
          const int at = at0 + 3 * S::PS * q;
          O[c][q] += Cb[0][q] * X[0][at] + Cb[1][q] * X[1][at] + Cb[2][q] * B[c][at];
        }
      }
    }
  };

  dl_up<LX, LXD>(sh[0], mats, g, 0);
  if constexpr (MODE == kFwd) {
    double C[3][PPT];
    if (on) {
#pragma unroll
      for (int q = 0; q < PPT; ++q) {
        const int at = at0 + 3 * S::PS * q;
        const double w3 = wij * w[k0 + 3 * q];
        double c9[9];
        metric(q, c9);
#pragma unroll
        for (int b = 0; b < 3; ++b)
          C[b][q] = w3 * (c9[3 * b] * B[0][at] + c9[3 * b + 1] * B[1][at] +
                          c9[3 * b + 2] * B[2][at]);
      }
    }
    convect(C);
  } else {
    // the first set's values at the thread's points: u' or the adjoint a
    double A[3][PPT];
    if (on) {
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int q = 0; q < PPT; ++q) A[d][q] = B[d][at0 + 3 * S::PS * q];
    }
    __syncthreads();
    dl_up<LX, LXD>(sh[0], mats, g, R3);
    if constexpr (MODE == kLin) {
      double C[3][PPT], Cp[3][PPT];
      if (on) {
#pragma unroll
        for (int q = 0; q < PPT; ++q) {
          const int at = at0 + 3 * S::PS * q;
          const double w3 = wij * w[k0 + 3 * q];
          double c9[9];
          metric(q, c9);
#pragma unroll
          for (int b = 0; b < 3; ++b) {
            C[b][q] = w3 * (c9[3 * b] * B[0][at] + c9[3 * b + 1] * B[1][at] +
                            c9[3 * b + 2] * B[2][at]);
            Cp[b][q] = w3 * (c9[3 * b] * A[0][q] + c9[3 * b + 1] * A[1][q] +
                             c9[3 * b + 2] * A[2][q]);
          }
        }
      }
      convect(Cp);
      // u' again for its own gradients
      if (t < R3) dl_row<LX>(g, a0, a1, a2, eb, t);
      __syncthreads();
      dl_up<LX, LXD>(sh[0], mats, g, 0);
      convect(C);
    } else {
      // E_b along the thread's line, the adjoint velocity through X
      double E[LXD];
#pragma unroll
      for (int l = 0; l < LXD; ++l) E[l] = 0.0;
      if (on) {
#pragma unroll
        for (int q = 0; q < PPT; ++q) {
          X[0][at0 + 3 * S::PS * q] = A[0][q];
          X[1][at0 + 3 * S::PS * q] = A[1][q];
        }
      }
      __syncthreads();
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        if (d == 2) {
          __syncthreads();
          if (on) {
#pragma unroll
            for (int q = 0; q < PPT; ++q) X[0][at0 + 3 * S::PS * q] = A[2][q];
          }
          __syncthreads();
        }
        if (on) {
          double in[LXD], out[LXD];
#pragma unroll
          for (int l = 0; l < LXD; ++l) in[l] = B[d][lb + l * ls];
          dl_apply<LXD, LXD>(mats + M::Dg, in, out);
          const double* a = X[d == 1 ? 1 : 0] + lb;
#pragma unroll
          for (int l = 0; l < LXD; ++l) E[l] += a[l * ls] * out[l];
        }
      }
      __syncthreads();
      // U at the thread's points, E_b in its place
      double U[3][PPT];
      if (on) {
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
          for (int q = 0; q < PPT; ++q) U[d][q] = B[d][at0 + 3 * S::PS * q];
      }
      __syncthreads();
      if (on) {
        double* o = B[db] + lb;
#pragma unroll
        for (int l = 0; l < LXD; ++l) o[l * ls] = E[l];
      }
      __syncthreads();
      if (on) {
#pragma unroll
        for (int q = 0; q < PPT; ++q) {
          const int at = at0 + 3 * S::PS * q;
          const double w3 = wij * w[k0 + 3 * q];
          double c9[9];
          metric(q, c9);
#pragma unroll
          for (int c = 0; c < 3; ++c)
            O[c][q] = w3 * (c9[c] * B[0][at] + c9[3 + c] * B[1][at] + c9[6 + c] * B[2][at]);
#pragma unroll
          for (int b = 0; b < 3; ++b)
            B[b][at] = w3 * (c9[3 * b] * U[0][q] + c9[3 * b + 1] * U[1][q] +
                             c9[3 * b + 2] * U[2][q]);
          X[0][at] = A[0][q];
          X[1][at] = A[1][q];
        }
      }
      __syncthreads();
      // C_b along the thread's line; then the weak term of each component
      double C[LXD];
      if (on) {
#pragma unroll
        for (int l = 0; l < LXD; ++l) C[l] = B[db][lb + l * ls];
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if (on) {
          const double* a = X[c == 1 ? 1 : 0] + lb;
          double in[LXD], out[LXD];
#pragma unroll
          for (int l = 0; l < LXD; ++l) in[l] = a[l * ls] * C[l];
          dl_apply<LXD, LXD>(mats + M::DgT, in, out);
          double* o = B[db] + lb;
#pragma unroll
          for (int l = 0; l < LXD; ++l) o[l * ls] = out[l];
        }
        __syncthreads();
        if (on) {
#pragma unroll
          for (int q = 0; q < PPT; ++q) {
            const int at = at0 + 3 * S::PS * q;
            O[c][q] += B[0][at] + B[1][at] + B[2][at];
            if (c == 0) X[0][at] = A[2][q];
          }
        }
        __syncthreads();
      }
    }
  }

  // f = beta f - (J x J x J)^T O
  __syncthreads();
  if (on) {
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int q = 0; q < PPT; ++q) B[c][at0 + 3 * S::PS * q] = O[c][q];
  }
  const int fc = t / (LX * LX), fl = t % (LX * LX);
  double* f = (fc == 0 ? fx : fc == 1 ? fy : fz) + eb + (int64_t)LX * fl;
  double old[LX];
#pragma unroll
  for (int l = 0; l < LX; ++l) old[l] = 0.0;
  if (t < R3 && beta != 0.0) {
#pragma unroll
    for (int l = 0; l < LX; ++l) old[l] = f[l];
  }
  __syncthreads();
  const double* JT = mats + M::JT;
  if (on) {
    const int c = t / S::NL, l = t % S::NL;
    dl_line<LXD, LX>(JT, B[c] + l % LXD + S::RS * (l / LXD), S::PS);
  }
  __syncthreads();
  if (t < 3 * LXD * LX) {
    const int c = t / (LXD * LX), l = t % (LXD * LX);
    dl_line<LXD, LX>(JT, B[c] + l % LXD + S::PS * (l / LXD), S::RS);
  }
  __syncthreads();
  if (t < R3) {
    const double* p = B[fc] + S::RS * (fl % LX) + S::PS * (fl / LX);
    double in[LXD], out[LX];
#pragma unroll
    for (int l = 0; l < LXD; ++l) in[l] = p[l];
    dl_apply<LXD, LX>(JT, in, out);
#pragma unroll
    for (int l = 0; l < LX; ++l) f[l] = (beta == 0.0 ? 0.0 : beta * old[l]) - out[l];
  }
}

// GL metric: the GLL cofactors of every element (from the coordinates and
// the GLL derivative matrix) interpolated to the GL points.
template <int LX, int LXD>
__global__ void __launch_bounds__(dl_threads<LXD>())
    dealias_metric_k(double* __restrict__ cof, const double* __restrict__ x,
                     const double* __restrict__ y,
                     const double* __restrict__ z,
                     const double* __restrict__ dx,
                     const double* __restrict__ mats, int64_t ngl) {
  constexpr int NT = dl_threads<LXD>();
  constexpr int NP = LX * LX * LX, NPG = LXD * LXD * LXD, NS = LX * LX;
  __shared__ DlShared<LX, LXD, 1> sh;
  __shared__ double sx[3][NP];
  __shared__ double sc[9][NP];
  __shared__ double sdx[LX * LX];
  const int e = blockIdx.x;
  const int64_t eb = (int64_t)e * NP, gb = (int64_t)e * NPG;
  load_mats(sh, mats);
  for (int p = threadIdx.x; p < NP; p += NT) {
    sx[0][p] = x[eb + p];
    sx[1][p] = y[eb + p];
    sx[2][p] = z[eb + p];
  }
  for (int p = threadIdx.x; p < LX * LX; p += NT) sdx[p] = dx[p];
  __syncthreads();
  for (int p = threadIdx.x; p < NP; p += NT) {
    const int i = p % LX, j = (p / LX) % LX, k = p / NS;
    double dr[3] = {0, 0, 0}, ds[3] = {0, 0, 0}, dt[3] = {0, 0, 0};
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int m = 0; m < LX; ++m) {
        dr[a] += sdx[i * LX + m] * sx[a][k * NS + j * LX + m];
        ds[a] += sdx[j * LX + m] * sx[a][k * NS + m * LX + i];
        dt[a] += sdx[k * LX + m] * sx[a][m * NS + j * LX + i];
      }
    // c_r = x_s x x_t, c_s = x_t x x_r, c_t = x_r x x_s
    sc[0][p] = ds[1] * dt[2] - ds[2] * dt[1];
    sc[1][p] = ds[2] * dt[0] - ds[0] * dt[2];
    sc[2][p] = ds[0] * dt[1] - ds[1] * dt[0];
    sc[3][p] = dt[1] * dr[2] - dt[2] * dr[1];
    sc[4][p] = dt[2] * dr[0] - dt[0] * dr[2];
    sc[5][p] = dt[0] * dr[1] - dt[1] * dr[0];
    sc[6][p] = dr[1] * ds[2] - dr[2] * ds[1];
    sc[7][p] = dr[2] * ds[0] - dr[0] * ds[2];
    sc[8][p] = dr[0] * ds[1] - dr[1] * ds[0];
  }
  __syncthreads();
  for (int m = 0; m < 9; ++m) {
    for (int p = threadIdx.x; p < NP; p += NT) sh.t2[p] = sc[m][p];
    __syncthreads();
    interp_up(sh, sh.buf[0]);
    for (int p = threadIdx.x; p < NPG; p += NT)
      cof[m * ngl + gb + p] = sh.buf[0][p];
    __syncthreads();
  }
}

// ---- host: the 1-D rules -------------------------------------------------

// Gauss-Legendre nodes (ascending) and weights: Newton on the three-term
// recurrence of P_n.
void gauss_legendre(int n, std::vector<double>& z, std::vector<double>& w) {
  z.assign(n, 0.0);
  w.assign(n, 0.0);
  auto legendre = [n](double x, double& pn, double& dpn) {
    double p0 = 1.0, p1 = x;
    for (int k = 2; k <= n; ++k) {
      const double p2 = ((2.0 * k - 1.0) * x * p1 - (k - 1.0) * p0) / k;
      p0 = p1;
      p1 = p2;
    }
    pn = p1;
    dpn = n * (x * p1 - p0) / (x * x - 1.0);
  };
  for (int i = 0; i < n; ++i) {
    double x = std::cos(M_PI * (i + 0.75) / (n + 0.5)), pn, dpn;
    for (int it = 0; it < 100; ++it) {
      legendre(x, pn, dpn);
      const double step = pn / dpn;
      x -= step;
      if (std::fabs(step) < 1e-16) break;
    }
    legendre(x, pn, dpn);
    z[n - 1 - i] = x;
    w[n - 1 - i] = 2.0 / ((1.0 - x * x) * dpn * dpn);
  }
}

template <int LX, int LXD>
int dealias_run(const DealiasState* s, int mode, double* fx, double* fy,
                double* fz, const double* a0, const double* a1,
                const double* a2, const double* b0, const double* b1,
                const double* b2, double beta) {
  const dim3 grid(s->nelv), block(Dl<LX, LXD>::NT);
  switch (mode) {
    case kFwd:
      hipLaunchKernelGGL((dealias_k<LX, LXD, kFwd>), grid, block, 0, stream(),
                         fx, fy, fz, a0, a1, a2, b0, b1, b2, s->cof, s->mats,
                         s->ngl, beta);
      break;
    case kLin:
      hipLaunchKernelGGL((dealias_k<LX, LXD, kLin>), grid, block, 0, stream(),
                         fx, fy, fz, a0, a1, a2, b0, b1, b2, s->cof, s->mats,
                         s->ngl, beta);
      break;
    default:
      hipLaunchKernelGGL((dealias_k<LX, LXD, kAdj>), grid, block, 0, stream(),
                         fx, fy, fz, a0, a1, a2, b0, b1, b2, s->cof, s->mats,
                         s->ngl, beta);
  }
  NK_LAUNCHED();
  return kOk;
}

#define NK_DL_SWITCH(LXV, CALL_T)                  \
  switch (LXV) {                                   \
    case 4: { constexpr int L = 4, LD = 6; CALL_T; } \
    case 6: { constexpr int L = 6, LD = 9; CALL_T; } \
    case 8: { constexpr int L = 8, LD = 12; CALL_T; } \
    default: break;                                \
  }

int dealias_apply(void* st, int mode, void* fx, void* fy, void* fz,
                  const void* a0, const void* a1, const void* a2,
                  const void* b0, const void* b1, const void* b2,
                  double beta) {
  NK_INIT();
  auto* s = static_cast<DealiasState*>(st);
  NK_REQUIRE(s != nullptr, "null dealias state");
  if (s->nelv == 0) return kOk;
  NK_REQUIRE(fx && fy && fz && a0 && a1 && a2, "null field");
  NK_REQUIRE(mode == kFwd || (b0 && b1 && b2), "null base flow");
  auto* X = (double*)fx;
  auto* Y = (double*)fy;
  auto* Z = (double*)fz;
  auto* A0 = (const double*)a0;
  auto* A1 = (const double*)a1;
  auto* A2 = (const double*)a2;
  auto* B0 = (const double*)b0;
  auto* B1 = (const double*)b1;
  auto* B2 = (const double*)b2;
  NK_DL_SWITCH(s->lx, return (dealias_run<L, LD>(s, mode, X, Y, Z, A0, A1, A2,
                                                  B0, B1, B2, beta)));
  return fail_arg(__func__, "unsupported lx");
}

}  // namespace
}  // namespace nekoamd

using namespace nekoamd;

extern "C" {

int nekoamd_dealias_create(void** st, const void* x, const void* y,
                           const void* z, const void* dx, const int* lx,
                           const int* lxd, const int* nelv) {
  NK_INIT();
  NK_REQUIRE(st && lx && lxd && nelv, "null argument");
  NK_REQUIRE(*nelv >= 0, "nelv < 0");
  if (!(*lx == 4 || *lx == 6 || *lx == 8) || *lxd != 3 * *lx / 2) {
    set_error(__func__, "dealiasing supports lx in {4, 6, 8} with lxd = 3 lx / 2");
    return kErrUnsupported;
  }
  NK_REQUIRE(*nelv == 0 || (x && y && z && dx), "null coordinates");
  auto* s = new DealiasState;
  s->lx = *lx;
  s->lxd = *lxd;
  s->nelv = *nelv;
  s->n = (int64_t)*nelv * *lx * *lx * *lx;
  s->ngl = (int64_t)*nelv * *lxd * *lxd * *lxd;
  const int L = *lx, LD = *lxd;
  std::vector<double> zl(L), wl(L), dl(L * L), zg, wg;
  int rc = nekoamd_gll(lx, zl.data(), wl.data(), dl.data());
  if (rc != kOk) {
    delete s;
    return rc;
  }
  gauss_legendre(LD, zg, wg);
  // J[q*L + i] = l_i(zg_q); Dg[i*LD + j] = l'_j(zg_i) on the GL nodes
  std::vector<double> mats(2 * (LD * L + LD * LD) + LD);
  for (int q = 0; q < LD; ++q)
    for (int i = 0; i < L; ++i) {
      double v = 1.0;
      for (int k = 0; k < L; ++k)
        if (k != i) v *= (zg[q] - zl[k]) / (zl[i] - zl[k]);
      mats[q * L + i] = v;
    }
  std::vector<double> a(LD, 1.0);
  for (int i = 0; i < LD; ++i)
    for (int k = 0; k < LD; ++k)
      if (k != i) a[i] *= zg[i] - zg[k];
  double* Dg = mats.data() + LD * L;
  for (int i = 0; i < LD; ++i) {
    double d = 0.0;
    for (int j = 0; j < LD; ++j) {
      if (j == i) continue;
      Dg[i * LD + j] = (a[i] / a[j]) / (zg[i] - zg[j]);
      d += 1.0 / (zg[i] - zg[j]);
    }
    Dg[i * LD + i] = d;
  }
  for (int i = 0; i < LD; ++i) mats[LD * L + LD * LD + i] = wg[i];
  double* JT = Dg + LD * LD + LD;
  double* DgT = JT + L * LD;
  for (int q = 0; q < LD; ++q)
    for (int i = 0; i < L; ++i) JT[i * LD + q] = mats[q * L + i];
  for (int i = 0; i < LD; ++i)
    for (int q = 0; q < LD; ++q) DgT[i * LD + q] = Dg[q * LD + i];
  hipError_t e = hipMalloc(&s->mats, sizeof(double) * mats.size());
  if (e == hipSuccess && s->ngl > 0)
    e = hipMalloc(&s->cof, sizeof(double) * 9 * (size_t)s->ngl);
  if (e == hipSuccess)
    e = hipMemcpyAsync(s->mats, mats.data(), sizeof(double) * mats.size(),
                       hipMemcpyHostToDevice, stream());
  if (e == hipSuccess && s->nelv > 0) {
    auto* X = (const double*)x;
    auto* Y = (const double*)y;
    auto* Z = (const double*)z;
    auto* D = (const double*)dx;
    NK_DL_SWITCH(L, hipLaunchKernelGGL((dealias_metric_k<L, LD>),
                                       dim3(s->nelv), dim3(dl_threads<LD>()),
                                       0, stream(), s->cof, X, Y, Z, D,
                                       s->mats, s->ngl);
                 break);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(stream());
  if (e != hipSuccess) {
    if (s->cof) (void)hipFree(s->cof);
    if (s->mats) (void)hipFree(s->mats);
    delete s;
    return fail_hip(__func__, e);
  }
  *st = s;
  return kOk;
}

int nekoamd_dealias_free(void* st) {
  NK_INIT();
  auto* s = static_cast<DealiasState*>(st);
  if (!s) return kOk;
  NK_HIP(hipStreamSynchronize(stream()));
  if (s->cof) NK_HIP(hipFree(s->cof));
  if (s->mats) NK_HIP(hipFree(s->mats));
  delete s;
  return kOk;
}

int nekoamd_dealias_metric(const void* st, void* cof) {
  NK_INIT();
  auto* s = static_cast<const DealiasState*>(st);
  NK_REQUIRE(s && (cof || s->ngl == 0), "null argument");
  if (s->ngl == 0) return kOk;
  NK_HIP(hipMemcpyAsync(cof, s->cof, sizeof(double) * 9 * (size_t)s->ngl,
                        hipMemcpyDeviceToDevice, stream()));
  return kOk;
}

int nekoamd_dealias_advection(void* st, void* fx, void* fy, void* fz,
                              const void* u, const void* v, const void* w,
                              const double* beta) {
  NK_REQUIRE(beta != nullptr, "null beta");
  return dealias_apply(st, kFwd, fx, fy, fz, u, v, w, nullptr, nullptr,
                       nullptr, *beta);
}

int nekoamd_dealias_linear(void* st, void* fx, void* fy, void* fz,
                           const void* up, const void* vp, const void* wp,
                           const void* ub, const void* vb, const void* wb) {
  return dealias_apply(st, kLin, fx, fy, fz, up, vp, wp, ub, vb, wb, 1.0);
}

int nekoamd_dealias_adjoint(void* st, void* fx, void* fy, void* fz,
                            const void* ua, const void* va, const void* wa,
                            const void* ub, const void* vb, const void* wb) {
  return dealias_apply(st, kAdj, fx, fy, fz, ua, va, wa, ub, vb, wb, 1.0);
}

}  // extern "C"
