// mlp.hip -- the element-local network of the learned solver aid: BF16
// MFMA forward and backward, Adam, harvesting of (residual, solution) pairs
// from the solver, training and inference on gfx950.
//
// The reference has no learned component; its initial-guess accelerator is
// the projection of sources/adjoint/adjoint_pnpn.f90:102-105, :729-741
// (projection.hip).  This network adds one more direction to the initial
// guess of the pressure solve:
//   q = mask(mult QQ^T N(b)),  gamma = <q,b>/<q,Aq>,  x0 += gamma q,
//   b -= gamma A q
// where N maps, per element, the 512 values of the residual b and the 6
// face-neighbour means of b (all divided by the RMS of b) to 512 values:
//   518 -> 256 (SiLU) -> 256 (SiLU) -> 512.
// The Galerkin scaling makes the guess safe: it never increases the A-norm
// of the error, and gamma = 0 (no guess) when <q,Aq> <= 0.
//
// GEMMs: 64 x 64 output tiles of a 256-thread workgroup, K in steps of 64
// staged through two LDS buffers, v_mfma_f32_32x32x16_bf16 (four waves, one
// 32 x 32 tile each), FP32 accumulation.  Operands that are contiguous along
// the output dimension (both of the weight gradient's, the data gradient's
// weights) are transposed in registers on their way to LDS.  Bias, SiLU,
// SiLU', the loss and its gradient, the column sums of the bias gradients
// and the BF16 rounding are in the epilogues; the three weight gradients
// are one split-K launch.  A training gradient is seven launches and bound
// by their latency (7 GFLOP at 4096 rows is 6 us of matrix peak): 80 us at
// 4096 rows, 67 us at 256 and 177 us at 19200.  With 128 x 128 tiles
// transposed into LDS value by value (two-byte stores, four-way and worse
// bank conflicts), a launch per weight gradient, separate column-sum, loss
// and unpadding passes and no loads in flight across a step it was 348, 231
// and 652 us (23 launches).
// BF16 is stored as uint16_t and rounded to nearest-even by bit arithmetic.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "internal.h"
#include "nekoamd.h"
#include "reduce.h"

namespace nekoamd {

constexpr int kNP = 512;    // GLL values per element (lx = 8)
constexpr int kNIN = 518;   // inputs
constexpr int kKIN = 544;   // inputs padded to the K tile
constexpr int kHID = 256;
// GEMM tile; LDS rows of 72 halfwords (36 banks), so that the 16-byte
// accesses of 8 consecutive lanes, in rows or in every other row, fall into
// distinct banks.
constexpr int kBT = 64, kBK = 64, kLdsK = kBK + 8;
constexpr int kMaxSplit = 16;

// padded parameter layout (FP32): W1[256][544] b1 W2[256][256] b2
// W3[512][256] b3
constexpr int64_t kOffW1 = 0;
constexpr int64_t kOffB1 = kOffW1 + (int64_t)kHID * kKIN;
constexpr int64_t kOffW2 = kOffB1 + kHID;
constexpr int64_t kOffB2 = kOffW2 + (int64_t)kHID * kHID;
constexpr int64_t kOffW3 = kOffB2 + kHID;
constexpr int64_t kOffB3 = kOffW3 + (int64_t)kNP * kHID;
constexpr int64_t kNParPad = kOffB3 + kNP;
static_assert(NEKOAMD_MLP_NPARAM ==
                  kHID * kNIN + kHID + kHID * kHID + kHID + kNP * kHID + kNP,
              "parameter count");

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) {
  return __uint_as_float((uint32_t)h << 16);
}
__device__ __forceinline__ float silu(float z) {
  return z / (1.0f + __expf(-z));
}
__device__ __forceinline__ float dsilu(float z) {
  const float s = 1.0f / (1.0f + __expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

enum Epi { kFwdHidden, kFwdOut, kFwdLoss, kBwdData };

struct EpiArgs {
  const float* bias;  // forward
  float* zf;          // FwdHidden: Z (may be null)
  uint16_t* hb;       // FwdHidden: H; FwdLoss, BwdData: dZ
  const float* z;     // BwdData: the forward pre-activation; FwdLoss: targets
  float* yf;          // FwdOut (float output)
  double* yd;         // FwdOut (double output, scaled by *yscale)
  const double* yscale;  // FwdOut; FwdLoss: yscale[1] scales the targets
                         // (null: unscaled)
  float gscale;       // FwdLoss: 2 / (M 512)
  float* colpart;     // FwdLoss, BwdData: [tile row][ldc] column sums of dZ
  double* lpart;      // FwdLoss: one loss partial per workgroup
  int ldc;
};

// One operand's 64 x 64 tile on its way to LDS: 16 BF16 values per thread.
// KM false: the operand is P[row][ld] with k contiguous; a thread holds
// two 8-value pieces of rows.  KM true: P[k][ld] with the output dimension
// contiguous; a thread holds columns c0 + 2 (t % 32) and the next of the 8
// rows of k group t / 32 (4-byte loads, 128 bytes of a row per half wave),
// and the store turns them into two 8-value pieces along k.  Values past
// `rows` or kend are zero; K ranges are multiples of 8.
template <bool KM>
struct Stage {
  uint32_t v[8];
  __device__ __forceinline__ void load(const uint16_t* __restrict__ P, int ld,
                                       int c0, int rows, int k0, int kend) {
    const int t = threadIdx.x;
    if constexpr (KM) {
      const int c = c0 + 2 * (t & 31), k = k0 + 8 * (t >> 5);
      const bool in = c < rows && k < kend;
      const uint16_t* q = P + (int64_t)k * ld + c;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        v[j] = in ? *(const uint32_t*)(q + (int64_t)j * ld) : 0u;
    } else {
#pragma unroll
      for (int c2 = 0; c2 < 2; ++c2) {
        const int c = t + c2 * 256, r = c0 + (c >> 3), k = k0 + (c & 7) * 8;
        uint4 w = make_uint4(0, 0, 0, 0);
        if (r < rows && k < kend) w = *(const uint4*)(P + (int64_t)r * ld + k);
        v[4 * c2] = w.x;
        v[4 * c2 + 1] = w.y;
        v[4 * c2 + 2] = w.z;
        v[4 * c2 + 3] = w.w;
      }
    }
  }
  __device__ __forceinline__ void store(uint16_t* lds) const {
    const int t = threadIdx.x;
    if constexpr (KM) {
      uint32_t lo[4], hi[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        lo[j] = (v[2 * j] & 0xFFFFu) | (v[2 * j + 1] << 16);
        hi[j] = (v[2 * j] >> 16) | (v[2 * j + 1] & 0xFFFF0000u);
      }
      uint16_t* d = lds + 2 * (t & 31) * kLdsK + 8 * (t >> 5);
      *(uint4*)d = make_uint4(lo[0], lo[1], lo[2], lo[3]);
      *(uint4*)(d + kLdsK) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    } else {
#pragma unroll
      for (int c2 = 0; c2 < 2; ++c2) {
        const int c = t + c2 * 256;
        *(uint4*)(lds + (c >> 3) * kLdsK + (c & 7) * 8) =
            make_uint4(v[4 * c2], v[4 * c2 + 1], v[4 * c2 + 2], v[4 * c2 + 3]);
      }
    }
  }
};

// acc = this wave's 32 x 32 part of sum_k A[m0+.][k] B[n0+.][k], k in
// [kbeg, kend).  The next step's loads are in flight while a step is
// multiplied, one barrier per step: the launches of a training batch have
// one to four workgroups per CU, so nothing else hides the latency.
constexpr int kTileLds = 4 * kBT * kLdsK;  // halfwords: two buffers of A and B
template <bool AKM, bool BKM>
__device__ __forceinline__ f32x16 tile_mma(const uint16_t* __restrict__ A,
                                           int lda, int m0, int M,
                                           const uint16_t* __restrict__ B,
                                           int ldb, int n0, int N, int kbeg,
                                           int kend, uint16_t* lds) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int ra = ((w >> 1) * 32 + (lane & 31)) * kLdsK + (lane >> 5) * 8;
  const int rb = ((w & 1) * 32 + (lane & 31)) * kLdsK + (lane >> 5) * 8;
  f32x16 acc;
#pragma unroll
  for (int a = 0; a < 16; ++a) acc[a] = 0.0f;
  Stage<AKM> sa;
  Stage<BKM> sb;
  sa.load(A, lda, m0, M, kbeg, kend);
  sb.load(B, ldb, n0, N, kbeg, kend);
  int buf = 0;
  for (int k0 = kbeg; k0 < kend; k0 += kBK) {
    uint16_t* la = lds + buf * 2 * kBT * kLdsK;
    uint16_t* lb = la + kBT * kLdsK;
    sa.store(la);
    sb.store(lb);
    // the buffer of the step before is written again only after this barrier
    // of the next step, which every wave reaches when done reading it
    __syncthreads();
    if (k0 + kBK < kend) {
      sa.load(A, lda, m0, M, k0 + kBK, kend);
      sb.load(B, ldb, n0, N, k0 + kBK, kend);
    }
#pragma unroll
    for (int ks = 0; ks < kBK; ks += 16) {
      const bf16x8 a = __builtin_bit_cast(bf16x8, *(const uint4*)(la + ra + ks));
      const bf16x8 b = __builtin_bit_cast(bf16x8, *(const uint4*)(lb + rb + ks));
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
    }
    buf ^= 1;
  }
  return acc;
}

// Row of accumulator value a: D[row][col], col = lane % 32,
// row = 8 (a / 4) + 4 (lane / 32) + a % 4.
__device__ __forceinline__ int acc_row(int a, int lane) {
  return 8 * (a >> 2) + 4 * (lane >> 5) + (a & 3);
}

// C[M,N] = sum_k A[m][k] B[n][k] (BKM: B[k][n]) with the epilogue EPI.
// Tiles of 64 x 64 for all M: at 4096 rows the widest layer has 512
// workgroups, at 32768 rows the narrow ones 2048.  The forward pass takes
// 22, 24 and 79 us at 256, 4096 and 32768 rows (29, 32 and 79 us with a K
// step of 32 and no loads in flight across it).
template <bool BKM, int EPI>
__global__ void __launch_bounds__(256)
    gemm_bf16_k(int M, int N, int K, const uint16_t* __restrict__ A, int lda,
                const uint16_t* __restrict__ B, int ldb, EpiArgs ep) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[kTileLds];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int m0 = blockIdx.x * kBT, n0 = blockIdx.y * kBT;
  const int rw = m0 + (w >> 1) * 32, col = n0 + (w & 1) * 32 + (lane & 31);
  f32x16 acc = tile_mma<false, BKM>(A, lda, m0, M, B, ldb, n0, N, 0, K, lds);
  if constexpr (EPI == kFwdHidden || EPI == kFwdOut) {
    if (col >= N) return;
    const float bias = ep.bias[col];
#pragma unroll
    for (int a = 0; a < 16; ++a) {
      const int row = rw + acc_row(a, lane);
      if (row >= M) continue;
      const int64_t o = (int64_t)row * ep.ldc + col;
      const float z = acc[a] + bias;
      if constexpr (EPI == kFwdHidden) {
        if (ep.zf) ep.zf[o] = z;
        ep.hb[o] = f2bf(silu(z));
      } else {
        if (ep.yf) ep.yf[o] = z;
        if (ep.yd) ep.yd[o] = (double)z * ep.yscale[0];
      }
    }
  } else {
    // dZ: FwdLoss d(loss)/dY of Y = acc + bias against the targets, BwdData
    // acc * silu'(Z); stored in BF16, its column sums over the tile's 64
    // rows taken from the FP32 values.  N is a multiple of the tile here.
    float z[16];
#pragma unroll
    for (int a = 0; a < 16; ++a) {
      const int row = min(rw + acc_row(a, lane), M - 1);
      z[a] = ep.z[(int64_t)row * ep.ldc + col];
    }
    const float bias = EPI == kFwdLoss ? ep.bias[col] : 0.0f;
    const float inv =
        EPI == kFwdLoss && ep.yscale != nullptr ? (float)ep.yscale[1] : 1.0f;
    double loss = 0.0;
    float cs = 0.0f;
#pragma unroll
    for (int a = 0; a < 16; ++a) {
      const int row = rw + acc_row(a, lane);
      if (row >= M) continue;
      float dz;
      if constexpr (EPI == kFwdLoss) {
        const float d = acc[a] + bias - z[a] * inv;
        loss += (double)d * (double)d;
        dz = ep.gscale * d;
      } else {
        dz = acc[a] * dsilu(z[a]);
      }
      ep.hb[(int64_t)row * ep.ldc + col] = f2bf(dz);
      cs += dz;
    }
    __shared__ float scol[2][kBT];
    __shared__ double sloss[4];
    cs += __shfl_xor(cs, 32, 64);
    if (lane < 32) scol[w >> 1][(w & 1) * 32 + lane] = cs;
    if constexpr (EPI == kFwdLoss) {
      loss = wave_sum(loss);
      if (lane == 0) sloss[w] = loss;
    }
    __syncthreads();
    if (threadIdx.x < kBT)
      ep.colpart[(int64_t)blockIdx.x * ep.ldc + n0 + threadIdx.x] =
          scol[0][threadIdx.x] + scol[1][threadIdx.x];
    if (EPI == kFwdLoss && threadIdx.x == 0)
      ep.lpart[blockIdx.y * gridDim.x + blockIdx.x] =
          (sloss[0] + sloss[1]) + (sloss[2] + sloss[3]);
  }
}

// The three weight gradients dW_l = dZ_l^T H_{l-1}, split over the rows:
// workgroup (tile, z) sums rows [z kz, (z+1) kz) of one 64 x 64 tile of one
// layer into ws[z] (the padded parameter layout).  One launch for all three:
// each alone has 16 to 36 tiles for 256 CUs.
struct WgradArgs {
  const uint16_t* dz[3];  // [M][rows[l]]
  const uint16_t* h[3];   // [M][cols[l]]
};
constexpr int kWgTiles1 = (kHID / kBT) * ((kKIN + kBT - 1) / kBT);
constexpr int kWgTiles2 = (kHID / kBT) * (kHID / kBT);
constexpr int kWgTiles3 = (kNP / kBT) * (kHID / kBT);
constexpr int kWgTiles = kWgTiles1 + kWgTiles2 + kWgTiles3;

__global__ void __launch_bounds__(256)
    mlp_wgrad_k(int M, int kz, WgradArgs v, float* __restrict__ ws) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[kTileLds];
  int tile = blockIdx.x, l = 0;
  int64_t off = kOffW1;
  if (tile >= kWgTiles1 + kWgTiles2) {
    tile -= kWgTiles1 + kWgTiles2;
    l = 2;
    off = kOffW3;
  } else if (tile >= kWgTiles1) {
    tile -= kWgTiles1;
    l = 1;
    off = kOffW2;
  }
  const int rows = l == 2 ? kNP : kHID, cols = l == 0 ? kKIN : kHID;
  const int m0 = tile % (rows / kBT) * kBT, n0 = tile / (rows / kBT) * kBT;
  const int kbeg = blockIdx.y * kz, kend = min(M, kbeg + kz);
  const f32x16 acc = tile_mma<true, true>(v.dz[l], rows, m0, rows, v.h[l],
                                          cols, n0, cols, kbeg, kend, lds);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int col = n0 + (w & 1) * 32 + (lane & 31);
  if (col >= cols) return;
  float* o = ws + (int64_t)blockIdx.y * kNParPad + off + col;
#pragma unroll
  for (int a = 0; a < 16; ++a)
    o[(int64_t)(m0 + (w >> 1) * 32 + acc_row(a, lane)) * cols] = acc[a];
}

// The gradient from its partial sums: weights over the nz row splits of ws,
// biases over the nt tile rows of cp ([nt][512] b3, then [nt][256] b2 and
// b1), acc[0] = (accum ? acc[0] : 0) + the np loss partials, each in a fixed
// order.  g: padded layout (the padding columns of W1 zero); out: unpadded
// (may be null).
constexpr int kFinW = (int)((kNParPad - (2 * kHID + kNP)) / 4 + 255) / 256;
constexpr int kFinB = (2 * kHID + kNP) / 16;
__global__ void __launch_bounds__(256)
    mlp_grad_fin_k(const float* __restrict__ ws, int nz,
                   const float* __restrict__ cp, int nt,
                   const double* __restrict__ lpart, int np, int accum,
                   double* __restrict__ acc, float* __restrict__ g,
                   float* __restrict__ out) {
  __shared__ float sc[256];
  __shared__ double sh[256 / 64];
  const int t = threadIdx.x, b = blockIdx.x;
  constexpr int64_t kPad = (int64_t)kHID * (kKIN - kNIN);
  if (b < kFinW) {
    // the i-th group of 4 weights, b1 and b2 left out
    int64_t i = 4 * ((int64_t)b * 256 + t);
    if (i >= kOffB1) i += kHID;
    if (i >= kOffB2) i += kHID;
    if (i >= kOffB3) return;
    float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 4
    for (int z = 0; z < nz; ++z) {
      const float4 v = *(const float4*)(ws + (int64_t)z * kNParPad + i);
      s.x += v.x;
      s.y += v.y;
      s.z += v.z;
      s.w += v.w;
    }
    float q[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t p = i + j;
      if (p < kOffB1) {
        const int64_t r = p / kKIN, c = p % kKIN;
        if (c >= kNIN) q[j] = 0.0f;
        else if (out) out[r * kNIN + c] = q[j];
      } else if (out) {
        out[p - kPad] = q[j];
      }
    }
    *(float4*)(g + i) = make_float4(q[0], q[1], q[2], q[3]);
  } else if (b < kFinW + kFinB) {
    // 16 columns, 16 threads each over the tile rows
    const int c0 = (b - kFinW) * 16, c = c0 + (t & 15), ch = t >> 4;
    const float* p = cp + c;  // b3
    int ld = kNP;
    int64_t o = kOffB3 + c;
    if (c0 >= kNP + kHID) {
      p = cp + (int64_t)nt * (kNP + kHID) + (c - kNP - kHID);
      ld = kHID;
      o = kOffB1 + (c - kNP - kHID);
    } else if (c0 >= kNP) {
      p = cp + (int64_t)nt * kNP + (c - kNP);
      ld = kHID;
      o = kOffB2 + (c - kNP);
    }
    float s = 0.0f;
#pragma unroll 4
    for (int r = ch; r < nt; r += 16) s += p[(int64_t)r * ld];
    sc[t] = s;
    __syncthreads();
    if (t < 16) {
      float q = 0.0f;
#pragma unroll
      for (int k = 0; k < 16; ++k) q += sc[k * 16 + t];
      g[o] = q;
      if (out) out[o - kPad] = q;
    }
  } else {
    const double s = sum_partials<256>(lpart, np, sh);
    if (t == 0) acc[0] = (accum ? acc[0] : 0.0) + s;
  }
}

// ---------------------------------------------------------------------------
// features, targets, scales

// part[b] = partial sum of u^2 over block b's share (fixed order).
__global__ void __launch_bounds__(kRedBlock)
    mlp_sumsq_k(int64_t n, const double* __restrict__ u,
                double* __restrict__ part) {
  __shared__ double sh[kRedBlock / 64];
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kRedBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kRedBlock)
    s += u[i] * u[i];
  s = block_sum<kRedBlock>(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// sc[0] = RMS = sqrt(sum/n), sc[1] = 1/RMS (1 when the field is zero).
__global__ void __launch_bounds__(kFinBlock)
    mlp_rms_fin_k(const double* __restrict__ part, int np, double n,
                  double* __restrict__ sc) {
  __shared__ double sh[kFinBlock / 64];
  const double s = sum_partials<kFinBlock>(part, np, sh);
  if (threadIdx.x == 0) {
    const double r = sqrt(s / n);
    sc[0] = r > 0.0 ? r : 1.0;
    sc[1] = r > 0.0 ? 1.0 / r : 1.0;
  }
}

// mean[e] = mean of the element's 512 values of u.
__global__ void __launch_bounds__(256)
    mlp_mean_k(const double* __restrict__ u, double* __restrict__ mean) {
  __shared__ double sh[256 / 64];
  const int64_t e = blockIdx.x;
  double s = u[e * kNP + threadIdx.x] + u[e * kNP + 256 + threadIdx.x];
  s = block_sum<256>(s, sh);
  if (threadIdx.x == 0) mean[e] = s * (1.0 / kNP);
}

// X[e][0..512) = bf16(u_e / s), X[e][512+k] = bf16(mean[nb] / s), rest 0.
__global__ void __launch_bounds__(64)
    mlp_features_k(const double* __restrict__ u,
                   const double* __restrict__ mean,
                   const int32_t* __restrict__ nbr,
                   const double* __restrict__ sc, uint16_t* __restrict__ X) {
  const int64_t e = blockIdx.x;
  const int t = threadIdx.x;
  const double inv = sc[1];
  uint16_t* xe = X + e * kKIN;
  uint16_t h[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) h[j] = f2bf((float)(u[e * kNP + t * 8 + j] * inv));
  uint4 hv;
  memcpy(&hv, h, sizeof(hv));
  *(uint4*)(xe + t * 8) = hv;
  if (t < 32) {
    const int c = kNP + t;  // 512 .. 543
    uint16_t v = 0;
    if (t < 6) {
      const int j = nbr[e * 6 + t];
      v = j >= 0 ? f2bf((float)(mean[j] * inv)) : (uint16_t)0;
    }
    xe[c] = v;
  }
}

// T[i] = x[i] / s (FP32)
__global__ void __launch_bounds__(256)
    mlp_target_k(int64_t n, const double* __restrict__ x,
                 const double* __restrict__ sc, float* __restrict__ T) {
  const double inv = sc[1];
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * 256)
    T[i] = (float)(x[i] * inv);
}

// Adam on the padded FP32 parameters; refreshes the BF16 weight copies.
// Padding entries have zero gradient and stay zero.
__global__ void __launch_bounds__(256)
    mlp_adam_k(float* __restrict__ th, const float* __restrict__ g,
               float* __restrict__ m, float* __restrict__ v, float lr,
               float b1, float b2, float c1, float c2, float eps,
               uint16_t* __restrict__ w1b, uint16_t* __restrict__ w2b,
               uint16_t* __restrict__ w3b) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < kNParPad;
       i += (int64_t)gridDim.x * 256) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float t = th[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    th[i] = t;
    if (i < kOffB1)
      w1b[i - kOffW1] = f2bf(t);
    else if (i >= kOffW2 && i < kOffB2)
      w2b[i - kOffW2] = f2bf(t);
    else if (i >= kOffW3 && i < kOffB3)
      w3b[i - kOffW3] = f2bf(t);
  }
}

__global__ void __launch_bounds__(256)
    mlp_tobf16_k(int64_t n, const float* __restrict__ a,
                 uint16_t* __restrict__ b) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * 256)
    b[i] = f2bf(a[i]);
}

__global__ void __launch_bounds__(256)
    mlp_axpy_k(int64_t n, double* __restrict__ y, const double* __restrict__ x,
               const double* __restrict__ a) {
  const double g = a[0];
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * 256)
    y[i] += g * x[i];
}

__global__ void __launch_bounds__(256)
    mlp_mulmask_k(int64_t n, double* __restrict__ q,
                  const double* __restrict__ mult) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * 256)
    q[i] *= mult[i];
}

// part = partials of {<q,b>_mult, <q,aq>_mult, <b,b>_mult}
__global__ void __launch_bounds__(kRedBlock)
    mlp_dots_k(int64_t n, const double* __restrict__ q,
               const double* __restrict__ b, const double* __restrict__ aq,
               const double* __restrict__ mult, double* __restrict__ part) {
  __shared__ double sh[kRedBlock / 64];
  double s0 = 0.0, s1 = 0.0, s2 = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kRedBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kRedBlock) {
    const double m = mult[i];
    s0 += m * q[i] * b[i];
    s1 += m * q[i] * aq[i];
    s2 += m * b[i] * b[i];
  }
  s0 = block_sum<kRedBlock>(s0, sh);
  s1 = block_sum<kRedBlock>(s1, sh);
  s2 = block_sum<kRedBlock>(s2, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = s0;
    part[kRedGrid + blockIdx.x] = s1;
    part[2 * kRedGrid + blockIdx.x] = s2;
  }
}

// sc[0..2] = the three sums; sc[3] = gamma = <q,b>/<q,aq> (0 unless
// <q,aq> > 0 and the result is finite).
__global__ void __launch_bounds__(kFinBlock)
    mlp_gamma_k(const double* __restrict__ part, int np,
                double* __restrict__ sc) {
  __shared__ double sh[kFinBlock / 64];
  const double qb = sum_partials<kFinBlock>(part, np, sh);
  const double qaq = sum_partials<kFinBlock>(part + kRedGrid, np, sh);
  const double bb = sum_partials<kFinBlock>(part + 2 * kRedGrid, np, sh);
  if (threadIdx.x == 0) {
    sc[0] = qb;
    sc[1] = qaq;
    sc[2] = bb;
    const double g = qaq > 0.0 ? qb / qaq : 0.0;
    sc[3] = isfinite(g) ? g : 0.0;
    sc[4] = -sc[3];
  }
}

// part[b] = partial sum of T^2 (FP32 values, FP64 sums)
__global__ void __launch_bounds__(kRedBlock)
    mlp_sumsq_f_k(int64_t n, const float* __restrict__ u,
                  double* __restrict__ part) {
  __shared__ double sh[kRedBlock / 64];
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kRedBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kRedBlock)
    s += (double)u[i] * (double)u[i];
  s = block_sum<kRedBlock>(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// ---------------------------------------------------------------------------
struct MlpState {
  int nelv = 0, nx = 0, ny = 0, nz = 0;
  int64_t n = 0;
  int cap = 0, npairs = 0, next = 0;
  int64_t adam_t = 0;
  int32_t* nbr = nullptr;
  float *th = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
  uint16_t *w1b = nullptr, *w2b = nullptr, *w3b = nullptr;
  // training set: X [cap*nelv][544] bf16, T [cap*nelv][512] f32
  uint16_t* Xd = nullptr;
  float* Td = nullptr;
  // per-batch work (rows = max(batch, nelv))
  int rows = 0;
  uint16_t *xb = nullptr, *h1 = nullptr, *h2 = nullptr, *dzb = nullptr;
  float *z1 = nullptr, *z2 = nullptr;
  float* ws = nullptr;     // kMaxSplit padded parameter sets: split-K partials
  float* cpart = nullptr;  // [tile row][512 + 256 + 256] column sums of dZ
  double* lpart = nullptr; // [tile row][512 / 64] loss partials
  double* mean = nullptr;  // nelv
  double* sc = nullptr;    // scalars: [0..1] rms/inv of the input field,
                           // [2..3] target scale, [8..12] guess dots/gamma
  double* part = nullptr;  // 3 * kRedGrid
  double* q = nullptr;     // n: the guess direction
  double* aq = nullptr;    // n
  double* bsave = nullptr; // n: residual kept for harvesting
  bool applied = false, saved = false;
  double* host = nullptr;  // pinned, 16
};

static MlpState* as_mlp(void* p) { return (MlpState*)p; }

template <bool BKM, int EPI>
static int gemm(int M, int N, int K, const uint16_t* A, int lda,
                const uint16_t* B, int ldb, const EpiArgs& ep) {
  if (M <= 0) return kOk;
  dim3 grid((M + kBT - 1) / kBT, (N + kBT - 1) / kBT);
  hipLaunchKernelGGL((gemm_bf16_k<BKM, EPI>), grid, dim3(256), 0, stream(), M,
                     N, K, A, lda, B, ldb, ep);
  NK_LAUNCHED();
  return kOk;
}

// The two hidden layers over M rows of X into the state's work buffers.
static int forward_hidden(MlpState* s, const uint16_t* X, int M, bool keep_z) {
  EpiArgs e{};
  e.bias = s->th + kOffB1;
  e.zf = keep_z ? s->z1 : nullptr;
  e.hb = s->h1;
  e.ldc = kHID;
  const int rc =
      gemm<false, kFwdHidden>(M, kHID, kKIN, X, kKIN, s->w1b, kKIN, e);
  if (rc) return rc;
  e.bias = s->th + kOffB2;
  e.zf = keep_z ? s->z2 : nullptr;
  e.hb = s->h2;
  return gemm<false, kFwdHidden>(M, kHID, kHID, s->h1, kHID, s->w2b, kHID, e);
}

static int forward(MlpState* s, const uint16_t* X, int M, float* yf,
                   double* yd, const double* yscale) {
  const int rc = forward_hidden(s, X, M, false);
  if (rc) return rc;
  EpiArgs o{};
  o.bias = s->th + kOffB3;
  o.yf = yf;
  o.yd = yd;
  o.yscale = yscale;
  o.ldc = kNP;
  return gemm<false, kFwdOut>(M, kNP, kHID, s->h2, kHID, s->w3b, kHID, o);
}

// Gradient of the batch (X, T) into s->g (padded layout) and out (unpadded,
// may be null); the loss sum into acc (added to it when accum).  ysc[1]:
// device scalar the targets are multiplied by (null: none).
static int backward(MlpState* s, const uint16_t* X, const float* T, int M,
                    const double* ysc, int accum, double* acc, float* out) {
  int rc = forward_hidden(s, X, M, true);
  if (rc) return rc;
  const int nt = (M + kBT - 1) / kBT;
  uint16_t* dz3 = s->dzb;
  uint16_t* dz2 = dz3 + (int64_t)M * kNP;
  uint16_t* dz1 = dz2 + (int64_t)M * kHID;
  EpiArgs e{};
  e.bias = s->th + kOffB3;
  e.z = T;
  e.hb = dz3;
  e.yscale = ysc;
  e.gscale = 2.0f / (float)((int64_t)M * kNP);
  e.colpart = s->cpart;
  e.lpart = s->lpart;
  e.ldc = kNP;
  rc = gemm<false, kFwdLoss>(M, kNP, kHID, s->h2, kHID, s->w3b, kHID, e);
  if (rc) return rc;
  EpiArgs d{};
  d.z = s->z2;
  d.hb = dz2;
  d.colpart = s->cpart + (int64_t)nt * kNP;
  d.ldc = kHID;
  rc = gemm<true, kBwdData>(M, kHID, kNP, dz3, kNP, s->w3b, kHID, d);
  if (rc) return rc;
  d.z = s->z1;
  d.hb = dz1;
  d.colpart += (int64_t)nt * kHID;
  rc = gemm<true, kBwdData>(M, kHID, kHID, dz2, kHID, s->w2b, kHID, d);
  if (rc) return rc;
  // row splits: at least one K step each, and no more than the partials'
  // buffer holds
  const int per = (nt + kMaxSplit - 1) / kMaxSplit;
  const int nz = (nt + per - 1) / per;
  WgradArgs v{{dz1, dz2, dz3}, {X, s->h1, s->h2}};
  hipLaunchKernelGGL(mlp_wgrad_k, dim3(kWgTiles, nz), dim3(256), 0, stream(),
                     M, per * kBK, v, s->ws);
  NK_LAUNCHED();
  hipLaunchKernelGGL(mlp_grad_fin_k, dim3(kFinW + kFinB + 1), dim3(256), 0,
                     stream(), s->ws, nz, s->cpart, nt, s->lpart,
                     nt * (kNP / kBT), accum, acc, s->g, out);
  NK_LAUNCHED();
  return kOk;
}

static int rms(MlpState* s, const double* u, double* out) {
  const int g = nk_grid(s->n, kRedBlock, kRedGrid);
  hipLaunchKernelGGL(mlp_sumsq_k, dim3(g), dim3(kRedBlock), 0, stream(), s->n,
                     u, s->part);
  NK_LAUNCHED();
  hipLaunchKernelGGL(mlp_rms_fin_k, dim3(1), dim3(kFinBlock), 0, stream(),
                     s->part, g, (double)s->n, out);
  NK_LAUNCHED();
  return kOk;
}

// X rows of one field (nelv rows) from u with scale sc[0..1].
static int make_features(MlpState* s, const double* u, const double* sc,
                         uint16_t* X) {
  hipLaunchKernelGGL(mlp_mean_k, dim3(s->nelv), dim3(256), 0, stream(), u,
                     s->mean);
  NK_LAUNCHED();
  hipLaunchKernelGGL(mlp_features_k, dim3(s->nelv), dim3(64), 0, stream(), u,
                     s->mean, s->nbr, sc, X);
  NK_LAUNCHED();
  return kOk;
}

template <typename T>
static T* dalloc(int64_t n, hipError_t& e) {
  T* p = nullptr;
  if (e == hipSuccess) e = hipMalloc((void**)&p, sizeof(T) * (n > 0 ? n : 1));
  return p;
}

static int refresh_bf16(MlpState* s) {
  hipLaunchKernelGGL(mlp_tobf16_k, dim3(nk_grid((int64_t)kHID * kKIN, 256)),
                     dim3(256), 0, stream(), (int64_t)kHID * kKIN,
                     s->th + kOffW1, s->w1b);
  NK_LAUNCHED();
  hipLaunchKernelGGL(mlp_tobf16_k, dim3(nk_grid((int64_t)kHID * kHID, 256)),
                     dim3(256), 0, stream(), (int64_t)kHID * kHID,
                     s->th + kOffW2, s->w2b);
  NK_LAUNCHED();
  hipLaunchKernelGGL(mlp_tobf16_k, dim3(nk_grid((int64_t)kNP * kHID, 256)),
                     dim3(256), 0, stream(), (int64_t)kNP * kHID,
                     s->th + kOffW3, s->w3b);
  NK_LAUNCHED();
  return kOk;
}

// q = mask(mult QQ^T N(r)): the network's element-local prediction for the
// residual r (its features scaled by the RMS of r, the output by it again),
// made continuous and zero on the mask -- the learned correction of the
// flexible CG (fcg.hip).  Uses the state's inference buffers; lx = 8.
int mlp_direction(void* mlp, int64_t n, const double* r, double* q,
                  const double* mult, void* gs, const int32_t* mask,
                  int64_t nmask) {
  MlpState* s = as_mlp(mlp);
  if (!s) return fail_arg("mlp_direction", "null network");
  if (s->n != n)
    return fail_arg("mlp_direction", "the network was made for another mesh");
  int rc = rms(s, r, s->sc);
  if (!rc) rc = make_features(s, r, s->sc, s->xb);
  if (!rc) rc = forward(s, s->xb, s->nelv, nullptr, q, s->sc);
  if (!rc) rc = gs_launch<double>(gs, q, NEKOAMD_GS_ADD, nullptr);
  if (rc) return rc;
  hipLaunchKernelGGL(mlp_mulmask_k, dim3(nk_grid(s->n, 256)), dim3(256), 0,
                     stream(), s->n, q, mult);
  NK_LAUNCHED();
  return bc_zero_launch<double>(q, mask, nmask, nullptr);
}

}  // namespace nekoamd

using namespace nekoamd;

extern "C" {

int nekoamd_mlp_create(void** mlp, const int* nx, const int* ny, const int* nz,
                       const int* lx, const int* capacity, const int* batch,
                       const int64_t* seed) {
  NK_INIT();
  NK_REQUIRE(mlp && nx && ny && nz && lx && capacity && batch && seed,
             "null argument");
  NK_REQUIRE(*lx == 8, "the network takes lx = 8 elements (512 GLL values)");
  NK_REQUIRE(*nx > 0 && *ny > 0 && *nz > 0, "empty mesh");
  NK_REQUIRE(*capacity >= 0 && *batch >= 32 && *batch % 32 == 0,
             "capacity >= 0 and batch a positive multiple of 32");
  MlpState* s = new MlpState();
  s->nx = *nx;
  s->ny = *ny;
  s->nz = *nz;
  s->nelv = *nx * *ny * *nz;
  s->n = (int64_t)s->nelv * kNP;
  s->cap = *capacity;
  s->rows = s->nelv > *batch ? s->nelv : *batch;
  const int64_t R = s->rows;
  const int64_t nt = (R + kBT - 1) / kBT;
  hipError_t e = hipSuccess;
  s->nbr = dalloc<int32_t>((int64_t)s->nelv * 6, e);
  s->th = dalloc<float>(kNParPad, e);
  s->g = dalloc<float>(kNParPad, e);
  s->m = dalloc<float>(kNParPad, e);
  s->v = dalloc<float>(kNParPad, e);
  s->w1b = dalloc<uint16_t>((int64_t)kHID * kKIN, e);
  s->w2b = dalloc<uint16_t>((int64_t)kHID * kHID, e);
  s->w3b = dalloc<uint16_t>((int64_t)kNP * kHID, e);
  s->Xd = dalloc<uint16_t>((int64_t)s->cap * s->nelv * kKIN, e);
  s->Td = dalloc<float>((int64_t)s->cap * s->nelv * kNP, e);
  s->xb = dalloc<uint16_t>(R * kKIN, e);
  s->h1 = dalloc<uint16_t>(R * kHID, e);
  s->h2 = dalloc<uint16_t>(R * kHID, e);
  s->dzb = dalloc<uint16_t>(R * (kNP + 2 * kHID), e);
  s->z1 = dalloc<float>(R * kHID, e);
  s->z2 = dalloc<float>(R * kHID, e);
  s->ws = dalloc<float>(kMaxSplit * kNParPad, e);
  s->cpart = dalloc<float>(nt * (kNP + 2 * kHID), e);
  s->lpart = dalloc<double>(nt * (kNP / kBT), e);
  s->mean = dalloc<double>(s->nelv, e);
  s->sc = dalloc<double>(16, e);
  s->part = dalloc<double>(3 * kRedGrid, e);
  s->q = dalloc<double>(s->n, e);
  s->aq = dalloc<double>(s->n, e);
  s->bsave = dalloc<double>(s->n, e);
  if (e == hipSuccess)
    e = hipHostMalloc((void**)&s->host, 16 * sizeof(double),
                      hipHostMallocDefault);
  if (e != hipSuccess) {
    nekoamd_mlp_free(s);
    return fail_hip(__func__, e);
  }
  // neighbour table of the x-fastest box numbering
  std::vector<int32_t> nb((size_t)s->nelv * 6);
  for (int el = 0; el < s->nelv; ++el) {
    const int ex = el % s->nx, ey = (el / s->nx) % s->ny,
              ez = el / (s->nx * s->ny);
    const int d[6][3] = {{-1, 0, 0}, {1, 0, 0}, {0, -1, 0},
                         {0, 1, 0},  {0, 0, -1}, {0, 0, 1}};
    for (int k = 0; k < 6; ++k) {
      const int jx = ex + d[k][0], jy = ey + d[k][1], jz = ez + d[k][2];
      const bool in = jx >= 0 && jx < s->nx && jy >= 0 && jy < s->ny &&
                      jz >= 0 && jz < s->nz;
      nb[(size_t)el * 6 + k] = in ? jx + s->nx * (jy + s->ny * jz) : -1;
    }
  }
  // initial weights U(-1/sqrt(fan_in), 1/sqrt(fan_in)), biases 0, padding 0
  std::vector<float> th((size_t)kNParPad, 0.0f);
  std::mt19937_64 rng((uint64_t)*seed);
  std::uniform_real_distribution<double> uni(-1.0, 1.0);
  for (int o = 0; o < kHID; ++o)
    for (int i = 0; i < kNIN; ++i)
      th[kOffW1 + (int64_t)o * kKIN + i] = (float)(uni(rng) / std::sqrt(518.0));
  for (int64_t i = 0; i < (int64_t)kHID * kHID; ++i)
    th[kOffW2 + i] = (float)(uni(rng) / 16.0);
  for (int64_t i = 0; i < (int64_t)kNP * kHID; ++i)
    th[kOffW3 + i] = (float)(uni(rng) / 16.0);
  e = hipMemcpy(s->nbr, nb.data(), nb.size() * 4, hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(s->th, th.data(), th.size() * 4, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemset(s->m, 0, kNParPad * 4);
  if (e == hipSuccess) e = hipMemset(s->v, 0, kNParPad * 4);
  if (e == hipSuccess) e = hipMemset(s->g, 0, kNParPad * 4);
  if (e != hipSuccess) {
    nekoamd_mlp_free(s);
    return fail_hip(__func__, e);
  }
  int rc = refresh_bf16(s);
  if (rc) {
    nekoamd_mlp_free(s);
    return rc;
  }
  *mlp = s;
  return kOk;
}

int nekoamd_mlp_free(void* mlp) {
  MlpState* s = as_mlp(mlp);
  if (!s) return kOk;
  if (initialised()) NK_HIP(hipStreamSynchronize(stream()));
  void* dev[] = {s->nbr, s->th,  s->g,    s->m,    s->v,  s->w1b, s->w2b,
                 s->w3b, s->Xd,  s->Td,   s->xb,   s->h1, s->h2,  s->dzb,
                 s->z1,  s->z2,  s->cpart, s->lpart, s->ws, s->mean, s->sc,
                 s->part, s->q,  s->aq,   s->bsave};
  for (void* p : dev)
    if (p) NK_HIP(hipFree(p));
  if (s->host) NK_HIP(hipHostFree(s->host));
  delete s;
  return kOk;
}

int nekoamd_mlp_get_params(void* mlp, float* out) {
  NK_INIT();
  MlpState* s = as_mlp(mlp);
  NK_REQUIRE(s && out, "null argument");
  std::vector<float> th((size_t)kNParPad);
  NK_HIP(hipStreamSynchronize(stream()));
  NK_HIP(hipMemcpy(th.data(), s->th, kNParPad * 4, hipMemcpyDeviceToHost));
  int64_t o = 0;
  for (int r = 0; r < kHID; ++r)
    for (int i = 0; i < kNIN; ++i) out[o++] = th[kOffW1 + (int64_t)r * kKIN + i];
  for (int64_t i = kOffB1; i < kNParPad; ++i) out[o++] = th[i];
  return kOk;
}

int nekoamd_mlp_set_params(void* mlp, const float* in) {
  NK_INIT();
  MlpState* s = as_mlp(mlp);
  NK_REQUIRE(s && in, "null argument");
  std::vector<float> th((size_t)kNParPad, 0.0f);
  int64_t o = 0;
  for (int r = 0; r < kHID; ++r)
    for (int i = 0; i < kNIN; ++i) th[kOffW1 + (int64_t)r * kKIN + i] = in[o++];
  for (int64_t i = kOffB1; i < kNParPad; ++i) th[i] = in[o++];
  NK_HIP(hipStreamSynchronize(stream()));
  NK_HIP(hipMemcpy(s->th, th.data(), kNParPad * 4, hipMemcpyHostToDevice));
  NK_HIP(hipMemset(s->m, 0, kNParPad * 4));
  NK_HIP(hipMemset(s->v, 0, kNParPad * 4));
  s->adam_t = 0;
  return refresh_bf16(s);
}

int nekoamd_mlp_forward(void* mlp, const void* X, const int* M, void* Y,
                        void* H1, void* H2) {
  NK_INIT();
  MlpState* s = as_mlp(mlp);
  NK_REQUIRE(s && X && M && Y, "null argument");
  NK_REQUIRE(*M >= 0 && *M <= s->rows, "M exceeds the work buffers");
  int rc = forward(s, (const uint16_t*)X, *M, (float*)Y, nullptr, nullptr);
  if (rc) return rc;
  if (H1)
    NK_HIP(hipMemcpyAsync(H1, s->h1, (size_t)*M * kHID * 2,
                          hipMemcpyDeviceToDevice, stream()));
  if (H2)
    NK_HIP(hipMemcpyAsync(H2, s->h2, (size_t)*M * kHID * 2,
                          hipMemcpyDeviceToDevice, stream()));
  return kOk;
}

int nekoamd_mlp_loss_grad(void* mlp, const void* X, const void* T,
                          const int* M, double* loss, void* g) {
  NK_INIT();
  MlpState* s = as_mlp(mlp);
  NK_REQUIRE(s && X && T && M && loss && g, "null argument");
  NK_REQUIRE(*M > 0 && *M <= s->rows && *M % 8 == 0,
             "M must be a positive multiple of 8 within the work buffers");
  int rc = backward(s, (const uint16_t*)X, (const float*)T, *M, nullptr, 0,
                    s->sc + 6, (float*)g);
  if (!rc) rc = to_host(s->host + 2, s->sc + 6, sizeof(double));
  if (rc) return rc;
  NK_HIP(hipStreamSynchronize(stream()));
  *loss = s->host[2] / ((double)*M * kNP);
  return kOk;
}

int nekoamd_mlp_harvest(void* mlp, const void* b, const void* x) {
  NK_INIT();
  MlpState* s = as_mlp(mlp);
  NK_REQUIRE(s && b && x, "null argument");
  if (s->cap == 0) return kOk;
  const int slot = s->next;
  uint16_t* X = s->Xd + (int64_t)slot * s->nelv * kKIN;
  float* T = s->Td + (int64_t)slot * s->n;
  int rc = rms(s, (const double*)b, s->sc);
  if (!rc) rc = make_features(s, (const double*)b, s->sc, X);
  if (rc) return rc;
  hipLaunchKernelGGL(mlp_target_k, dim3(nk_grid(s->n, 256)), dim3(256), 0,
                     stream(), s->n, (const double*)x, s->sc, T);
  NK_LAUNCHED();
  s->next = (s->next + 1) % s->cap;
  if (s->npairs < s->cap) ++s->npairs;
  return kOk;
}

int nekoamd_mlp_pairs(void* mlp, int* npairs) {
  MlpState* s = as_mlp(mlp);
  if (!s || !npairs) return fail_arg(__func__, "null argument");
  *npairs = s->npairs;
  return kOk;
}

int nekoamd_mlp_train(void* mlp, const int* epochs, const int* batch,
                      const float* lr, const int64_t* seed, double* loss_first,
                      double* loss_last) {
  NK_INIT();
  MlpState* s = as_mlp(mlp);
  NK_REQUIRE(s && epochs && batch && lr && seed && loss_first && loss_last,
             "null argument");
  NK_REQUIRE(*batch >= 32 && *batch % 32 == 0 && *batch <= s->rows,
             "batch must be a multiple of 32 within the work buffers");
  NK_REQUIRE(*epochs >= 1, "epochs must be positive");
  NK_REQUIRE(s->npairs > 0, "no harvested pairs");
  const int64_t S = (int64_t)s->npairs * s->nelv;
  const int B = *batch;
  const int64_t nb = S / B;
  NK_REQUIRE(nb > 0, "fewer samples than one batch");
  // target scale sc[2..3] = RMS of the stored targets and its inverse
  {
    const int64_t nt = S * kNP;
    const int g = nk_grid(nt, kRedBlock, kRedGrid);
    hipLaunchKernelGGL(mlp_sumsq_f_k, dim3(g), dim3(kRedBlock), 0, stream(),
                       nt, s->Td, s->part);
    NK_LAUNCHED();
    hipLaunchKernelGGL(mlp_rms_fin_k, dim3(1), dim3(kFinBlock), 0, stream(),
                       s->part, g, (double)nt, s->sc + 2);
    NK_LAUNCHED();
  }
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  std::mt19937_64 rng((uint64_t)*seed);
  std::vector<int64_t> order((size_t)nb);
  double* acc = s->sc + 6;
  for (int ep = 0; ep < *epochs; ++ep) {
    for (int64_t q = 0; q < nb; ++q) order[(size_t)q] = q;
    std::shuffle(order.begin(), order.end(), rng);
    for (int64_t q = 0; q < nb; ++q) {
      const int64_t r0 = order[(size_t)q] * B;
      const int rc = backward(s, s->Xd + r0 * kKIN, s->Td + r0 * kNP, B,
                              s->sc + 2, q > 0, acc, nullptr);
      if (rc) return rc;
      ++s->adam_t;
      const float c1 = 1.0f - powf(b1, (float)s->adam_t);
      const float c2 = 1.0f - powf(b2, (float)s->adam_t);
      hipLaunchKernelGGL(mlp_adam_k, dim3(nk_grid(kNParPad, 256)), dim3(256),
                         0, stream(), s->th, s->g, s->m, s->v, *lr, b1, b2, c1,
                         c2, eps, s->w1b, s->w2b, s->w3b);
      NK_LAUNCHED();
    }
    NK_HIP(hipMemcpyAsync(s->host, acc, sizeof(double), hipMemcpyDeviceToHost,
                          stream()));
    NK_HIP(hipStreamSynchronize(stream()));
    const double l = s->host[0] / ((double)nb * B * kNP);
    if (ep == 0) *loss_first = l;
    *loss_last = l;
  }
  return kOk;
}

// Learned initial guess of one solve.  save: keep b for harvesting in
// nekoamd_mlp_post; apply: q = mask(mult QQ^T N(b)), aq = mask(QQ^T A q),
// gamma = <q,b>/<q,aq>, b -= gamma aq.
int nekoamd_mlp_pre(void* mlp, void* b, const void* mult, void* gs,
                    const void* mask, const int64_t* nmask, const void* dx,
                    const void* h1, const void* h2, const void* g11,
                    const void* g12, const void* g13, const void* g22,
                    const void* g23, const void* g33, const void* B,
                    const int* lx, const int* ifh2, const int* apply,
                    const int* save, double* gamma) {
  NK_INIT();
  MlpState* s = as_mlp(mlp);
  NK_REQUIRE(s && b && mult && gs && nmask && dx && h1 && g11 && g12 && g13 &&
                 g22 && g23 && g33 && lx && ifh2 && apply && save && gamma,
             "null argument");
  NK_REQUIRE(*lx == 8, "lx must be 8");
  NK_REQUIRE(*nmask >= 0 && (*nmask == 0 || mask), "bad mask");
  NK_REQUIRE(!*ifh2 || (h2 && B), "ifh2 set but h2 or B is null");
  double* bd = (double*)b;
  const int64_t n = s->n;
  const int ge = nk_grid(n, 256);
  *gamma = 0.0;
  s->applied = false;
  s->saved = false;
  if (*save) {
    NK_HIP(hipMemcpyAsync(s->bsave, bd, sizeof(double) * n,
                          hipMemcpyDeviceToDevice, stream()));
    s->saved = true;
  }
  if (!*apply) return kOk;
  int rc = rms(s, bd, s->sc);
  if (!rc) rc = make_features(s, bd, s->sc, s->xb);
  if (!rc) rc = forward(s, s->xb, s->nelv, nullptr, s->q, s->sc);
  if (!rc) rc = gs_launch<double>(gs, s->q, NEKOAMD_GS_ADD, nullptr);
  if (rc) return rc;
  hipLaunchKernelGGL(mlp_mulmask_k, dim3(ge), dim3(256), 0, stream(), n, s->q,
                     (const double*)mult);
  NK_LAUNCHED();
  rc = bc_zero_launch<double>(s->q, (const int32_t*)mask, *nmask, nullptr);
  if (!rc)
    rc = ax_helm_launch<double, double>(
        s->aq, s->q, (const double*)dx, (const double*)h1, (const double*)h2,
        (const double*)g11, (const double*)g12, (const double*)g13,
        (const double*)g22, (const double*)g23, (const double*)g33,
        (const double*)B, 8, s->nelv, *ifh2 != 0, nullptr);
  if (!rc) rc = gs_launch<double>(gs, s->aq, NEKOAMD_GS_ADD, nullptr);
  if (!rc)
    rc = bc_zero_launch<double>(s->aq, (const int32_t*)mask, *nmask, nullptr);
  if (rc) return rc;
  const int gr = nk_grid(n, kRedBlock, kRedGrid);
  hipLaunchKernelGGL(mlp_dots_k, dim3(gr), dim3(kRedBlock), 0, stream(), n,
                     s->q, bd, s->aq, (const double*)mult, s->part);
  NK_LAUNCHED();
  hipLaunchKernelGGL(mlp_gamma_k, dim3(1), dim3(kFinBlock), 0, stream(),
                     s->part, gr, s->sc + 8);
  NK_LAUNCHED();
  hipLaunchKernelGGL(mlp_axpy_k, dim3(ge), dim3(256), 0, stream(), n, bd,
                     s->aq, s->sc + 12);
  NK_LAUNCHED();
  NK_HIP(hipMemcpyAsync(s->host, s->sc + 8, 4 * sizeof(double),
                        hipMemcpyDeviceToHost, stream()));
  NK_HIP(hipStreamSynchronize(stream()));
  *gamma = s->host[3];
  s->applied = true;
  return kOk;
}

// x += gamma q when a guess was applied; harvest (kept b, x) when asked and
// b was kept.
int nekoamd_mlp_post(void* mlp, void* x, const int* harvest) {
  NK_INIT();
  MlpState* s = as_mlp(mlp);
  NK_REQUIRE(s && x && harvest, "null argument");
  if (s->applied) {
    hipLaunchKernelGGL(mlp_axpy_k, dim3(nk_grid(s->n, 256)), dim3(256), 0,
                       stream(), s->n, (double*)x, s->q, s->sc + 11);
    NK_LAUNCHED();
    s->applied = false;
  }
  if (*harvest && s->saved) {
    s->saved = false;
    return nekoamd_mlp_harvest(mlp, s->bsave, x);
  }
  return kOk;
}

}  // extern "C"
