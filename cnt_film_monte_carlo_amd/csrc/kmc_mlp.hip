// kmc_mlp.hip -- learned surrogate of the first-order transfer rate.  No reference counterpart:
// it stands beside exciton_transfer::first_order (src/exciton_transfer/exciton_transfer.cpp:
// 380-441), which stays the fallback for flagged pairs.
//
// Network: 16 feature slots -> 4 hidden layers of 128 (SiLU) -> 1, predicting a normalised
// log10 rate.  All products run on the CDNA4 matrix cores as v_mfma_f32_32x32x16_bf16 with BF16
// operands and FP32 accumulation; master weights, biases and the output layer are FP32.
//
// A training step is three launches (activations and gradients of a tile stay on the chip):
//   k_mlp_rows   32 rows per workgroup through the whole network and back:
//                Z_l = H_{l-1} W_l + b_l, H_l = bf16(silu(Z_l)), y = H_3 . w4 + b4,
//                dy = 2 (y - t) / n, dZ_3 = bf16(dy w4 silu'(Z_3)),
//                dZ_{l-1} = bf16((dZ_l W_l^T) silu'(Z_{l-1})); leaves H_l and dZ_l, transposed
//   k_mlp_grads  dW_l = H_{l-1}^T dZ_l in splits over the batch, db_l, dw4, db4 in row blocks
//   k_mlp_update the splits' and blocks' sums in a fixed order, then Adam on the FP32 masters,
//                which refreshes both BF16 copies W_l and W_l^T.
// Inference: one fused kernel, one 32-pair tile per wave.  The BF16 weights (100 KB) sit in LDS,
// pre-arranged as MFMA A fragments; activations never leave registers because the hidden units
// of layers 1..3 are taken in the order in which the accumulator of the previous layer holds
// them (see k_pack), so a C tile becomes the next layer's B operand without any data movement.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <new>
#include <string>
#include <system_error>
#include <thread>
#include <vector>

#include "../../include/cntkmc.h"
#include "kmc_mlp.h"

namespace {

using bf16 = __bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int IN = KMC_MLP_IN, WD = KMC_MLP_WIDTH, NH = KMC_MLP_HIDDEN, NCLS = KMC_MLP_CLASSES;
constexpr int64_t NP = KMC_MLP_PARAMS;
constexpr int NBIN_PAIR = NCLS * NCLS;

__host__ __device__ constexpr int fan_in(int l) { return l == 0 ? IN : WD; }
// offsets in the FP32 parameter vector
__host__ __device__ constexpr int64_t w_off(int l) {
  return l == 0 ? 0 : w_off(l - 1) + (int64_t)fan_in(l - 1) * WD + WD;
}
__host__ __device__ constexpr int64_t b_off(int l) { return w_off(l) + (int64_t)fan_in(l) * WD; }
constexpr int64_t W4_OFF = w_off(NH), B4_OFF = W4_OFF + WD;
static_assert(B4_OFF + 1 == NP, "parameter layout");
// offsets of layer l in the BF16 weight copies (W_l, W_l^T and the packed inference layout)
__host__ __device__ constexpr int64_t q_off(int l) { return l == 0 ? 0 : q_off(l - 1) + (int64_t)fan_in(l - 1) * WD; }
constexpr int64_t NQ = q_off(NH);  // 51200 BF16 weights

// logistic function from the hardware exp2 and reciprocal (about 1 ulp each; the results feed
// BF16 operands), shared by training and inference so both evaluate the same network
__device__ __forceinline__ float sigmoid_f(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504088896341f * z));
}
__device__ __forceinline__ float silu_f(float z) { return z * sigmoid_f(z); }
__device__ __forceinline__ float dsilu_f(float z) {
  const float s = sigmoid_f(z);
  return s * (1.0f + z * (1.0f - s));
}
__device__ __forceinline__ f32x16 mfma32(const bf16x8& a, const bf16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------------------------------------
// features and residual-map bins (shared by host and device)
// ---------------------------------------------------------------------------------------------
struct domain_consts {
  double lo[3], hi[3], t_lo, t_hi, y_shift, y_scale;
};

__host__ __device__ inline double box_coord(double v, const domain_consts& d, int k) {
  const double c = fmin(fmax(v, d.lo[k]), d.hi[k]);
  return (2.0 * c - (d.lo[k] + d.hi[k])) / (d.hi[k] - d.lo[k]);
}
// Features 2..4: the box coordinates of z and of (a1, a2) taken with the sign that makes a2 > 0
// (a1 > 0 when a2 == 0); the a1/a2 box is symmetric, so clamping commutes with the flip.
__host__ __device__ inline void shift_features(double z, double a1, double a2, const domain_consts& d,
                                               float* f) {
  const double c1 = fmin(fmax(a1, d.lo[1]), d.hi[1]), c2 = fmin(fmax(a2, d.lo[2]), d.hi[2]);
  const bool flip = c2 < 0.0 || (c2 == 0.0 && c1 < 0.0);
  f[0] = (float)box_coord(z, d, 0);
  f[1] = (float)box_coord(flip ? -c1 : c1, d, 1);
  f[2] = (float)box_coord(flip ? -c2 : c2, d, 2);
}
__host__ __device__ inline double temp_feature(double T, const domain_consts& d) {
  return log(T / sqrt(d.t_lo * d.t_hi)) / log(sqrt(d.t_hi / d.t_lo));
}
__host__ __device__ inline double inv_temp_feature(double T, const domain_consts& d) {
  return (2.0 / T - (1.0 / d.t_lo + 1.0 / d.t_hi)) / (1.0 / d.t_lo - 1.0 / d.t_hi);
}
__host__ __device__ inline int bin_of(double u, int n) {  // u in [0, 1]
  const int b = (int)(u * n);
  return b < 0 ? 0 : b >= n ? n - 1 : b;
}
// Flattened (pair class, T, z, theta, max |a|) bin of one geometry.
__host__ __device__ inline int64_t bin_index(const int32_t* dims, int cd, int ca, double T, double th,
                                             double z, double a1, double a2, const domain_consts& d) {
  const double zc = fmin(fmax(z, d.lo[0]), d.hi[0]);
  const double c1 = fabs(fmin(fmax(a1, d.lo[1]), d.hi[1])), c2 = fabs(fmin(fmax(a2, d.lo[2]), d.hi[2]));
  const double amax = fmax(fmax(fabs(d.lo[1]), fabs(d.hi[1])), fmax(fabs(d.lo[2]), fabs(d.hi[2])));
  const int iT = bin_of((T - d.t_lo) / (d.t_hi - d.t_lo), dims[1]);
  const int iz = bin_of((zc - d.lo[0]) / (d.hi[0] - d.lo[0]), dims[2]);
  const int ith = bin_of(th / M_PI, dims[3]);
  const double ua = fmax(c1, c2) / amax;
  const int ia = bin_of(ua * ua, dims[4]);  // equal-area rings of the (a1, a2) square
  return ((((int64_t)(cd * NCLS + ca) * dims[1] + iT) * dims[2] + iz) * dims[3] + ith) * dims[4] + ia;
}

// ---------------------------------------------------------------------------------------------
// training kernels
// ---------------------------------------------------------------------------------------------
constexpr int TILE = 32;            // rows of one workgroup of k_mlp_rows
constexpr int K_SPLIT = 512;        // batch rows per split of the weight-gradient products
constexpr int LOSS_PARTS = 256;     // partial sums of the squared error
constexpr int COL_BLOCKS = 64;      // row blocks of the bias and output-layer gradients
constexpr int COLS = NH * WD + WD + 1;  // their columns: db_0..db_3, dw4, db4
constexpr int XS = WD + 8;          // LDS row of one sample's activations (padded: no bank conflicts)
constexpr int LEAVES = 72;          // LDS row of one sample's 64 products of the output unit

struct rows_args {
  int n_valid;            // rows beyond have no target
  const int32_t* idx;     // optional: batch row r is row idx[r] of X and tgt
  const bf16* X;          // [rows][IN]
  const float* tgt;
  float inv_n;
  const bf16 *Wtb, *Wb;   // W_l^T and W_l
  const float* prm;
  int64_t layer;          // elements of one layer of HT and DT
  bf16 *XT, *HT, *DT;     // X^T, H_l^T and dZ_l^T by tiles of 32 rows: [tile][unit][32]
  float *y, *dy, *err;
};

// A workgroup barrier for data in LDS: unlike __syncthreads it does not wait for the wave's
// global stores, which nothing in the kernel reads back.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ float lane_swap(float x) {  // the value of lane i ^ 1
  return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), 0xB1, 0xF, 0xF, true));
}

// One wave's 32 rows x 32 units as the accumulator holds them (register r of lane (h, c): row
// 8 (r / 4) + 4 h + r % 4, unit n = 32 wave + c): to LDS for the next layer's A operand (a
// sample's units side by side) and, transposed, to memory for the weight gradients.
__device__ __forceinline__ void put_tile(const bf16 (&v)[16], bf16 (*xa)[XS], int n, int h,
                                         bf16* __restrict__ T) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    bf16x4 p;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      xa[8 * q + 4 * h + j][n] = v[4 * q + j];
      p[j] = v[4 * q + j];
    }
    if (T) *reinterpret_cast<bf16x4*>(T + TILE * n + 8 * q + 4 * h) = p;
  }
}

__device__ __forceinline__ f32x16 layer_product(const bf16 (*xa)[XS], int c, int h,
                                                const bf16x8 (&w)[8]) {
  f32x16 acc = {};
#pragma unroll
  for (int kb = 0; kb < 8; ++kb)
    acc = mfma32(*reinterpret_cast<const bf16x8*>(&xa[c][16 * kb + 8 * h]), w[kb], acc);
  return acc;
}

// 32 rows per workgroup, 32 units of every layer per wave: the four waves exchange a layer's
// activations through LDS, and each holds its weight fragments (read from L2 ahead of their use),
// pre-activations and gradients in registers.  A batch of 8,192 rows is 256 workgroups, one per
// CU; what bounds it is the chain of seven layers, each eight MFMAs, an LDS exchange and sixteen
// SiLUs or their derivatives per lane.  The products run in the order of k (16 per MFMA) with the
// samples as A operand, and the output unit's 128 products are added in the order of a butterfly
// over 64 pairs of units, so that a batch's results do not depend on how it is tiled.
template <bool GRAD>
__global__ __launch_bounds__(256) void k_mlp_rows(rows_args g) {
  __shared__ __align__(16) bf16 xa[2][TILE][XS];
  __shared__ float leaf[TILE][LEAVES];
  __shared__ float s_d[TILE];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, h = lane >> 5, c = lane & 31;
  const int n = 32 * wv + c;
  const int64_t row0 = (int64_t)blockIdx.x * TILE, row = row0 + c;
  const int64_t src = g.idx ? g.idx[row] : row;
  const bf16x8 a0 = *reinterpret_cast<const bf16x8*>(g.X + src * IN + 8 * h);
  const bf16x8 w0 = *reinterpret_cast<const bf16x8*>(g.Wtb + (int64_t)n * IN + 8 * h);
  bf16x8 wf[3][8];
#pragma unroll
  for (int l = 1; l < NH; ++l)
#pragma unroll
    for (int kb = 0; kb < 8; ++kb)
      wf[l - 1][kb] = *reinterpret_cast<const bf16x8*>(g.Wtb + q_off(l) + (int64_t)n * WD + 16 * kb + 8 * h);
  if (GRAD && wv == 0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) g.XT[row0 * IN + TILE * (8 * h + e) + c] = a0[e];
  }
  float z[NH][16];
  bf16 v[16];
  f32x16 acc = {};
#pragma unroll
  for (int l = 0; l < NH; ++l) {
    if (l == 0) {
      acc = mfma32(a0, w0, acc);
    } else {
      lds_barrier();
      acc = layer_product(xa[(l - 1) & 1], c, h, wf[l - 1]);
    }
    const float bias = g.prm[b_off(l) + n];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      z[l][r] = acc[r] + bias;
      v[r] = (bf16)silu_f(z[l][r]);
    }
    if (l + 1 < NH || GRAD)
      put_tile(v, xa[l & 1], n, h, GRAD ? g.HT + l * g.layer + row0 * WD : nullptr);
  }
  // the weights of the way back, read while the output unit is summed
  bf16x8 wb[3][8];
  if (GRAD) {
#pragma unroll
    for (int l = 1; l < NH; ++l)
#pragma unroll
      for (int kb = 0; kb < 8; ++kb)
        wb[l - 1][kb] = *reinterpret_cast<const bf16x8*>(g.Wb + q_off(l) + (int64_t)n * WD + 16 * kb + 8 * h);
  }
  const float wa = g.prm[W4_OFF + n], wo = lane_swap(wa);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const float hv = (float)v[r], ho = lane_swap(hv);
    if (!(c & 1)) leaf[8 * (r >> 2) + 4 * h + (r & 3)][n >> 1] = fmaf(hv, wa, ho * wo);
  }
  lds_barrier();
  {
    const int s = threadIdx.x >> 3, p = threadIdx.x & 7;
    float u[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) u[q] = leaf[s][8 * q + p];
    float t = ((u[0] + u[4]) + (u[2] + u[6])) + ((u[1] + u[5]) + (u[3] + u[7]));
    t += __shfl_xor(t, 4, 64);
    t += __shfl_xor(t, 2, 64);
    t += __shfl_xor(t, 1, 64);
    const float yy = t + g.prm[B4_OFF];
    if (p == 0) {
      const int64_t q = row0 + s;
      g.y[q] = yy;
      if (GRAD) {
        const float e = q < g.n_valid ? yy - g.tgt[g.idx ? g.idx[q] : q] : 0.0f;
        const float d = 2.0f * e * g.inv_n;
        g.dy[q] = d;
        g.err[q] = e;
        s_d[s] = d;
      }
    }
  }
  if (!GRAD) return;
  lds_barrier();
#pragma unroll
  for (int r = 0; r < 16; ++r)
    v[r] = (bf16)(s_d[8 * (r >> 2) + 4 * h + (r & 3)] * wa * dsilu_f(z[NH - 1][r]));
  put_tile(v, xa[0], n, h, g.DT + (NH - 1) * g.layer + row0 * WD);
#pragma unroll
  for (int l = NH - 1; l >= 1; --l) {
    lds_barrier();
    acc = layer_product(xa[(NH - 1 - l) & 1], c, h, wb[l - 1]);
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = (bf16)(acc[r] * dsilu_f(z[l - 1][r]));
    put_tile(v, xa[(NH - l) & 1], n, h, g.DT + (l - 1) * g.layer + row0 * WD);
  }
}

struct grads_args {
  int nb, nz;             // rows (a multiple of 128) and splits of K_SPLIT rows
  int64_t layer;
  const bf16 *XT, *HT, *DT;
  const float *dy, *err;
  float* part;            // weight layer l: nz q_off(l) + [nz][fan_in][WD]
  float* cpart;           // [COL_BLOCKS][COLS]
  double* lpart;          // [LOSS_PARTS]
};

// Blocks [0, 13 nz): dW tiles.  A wave takes 32 x 32 weights over one split's rows, 16 per MFMA in
// row order, both operands 16 contiguous bytes of a transposed array per lane; layer 0 has one
// 32-row tile (16 features), the others four.  Then 3 COL_BLOCKS blocks of column sums (a thread
// per column, even and odd rows apart) and one block for the squared error.  832 waves and 192
// small blocks at 8,192 rows: bound by the latency of a split's chain of 32 MFMAs and its loads.
__global__ __launch_bounds__(256) void k_mlp_grads(grads_args g) {
#pragma clang fp contract(off)
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6, h = lane >> 5, c = lane & 31;
  int b = blockIdx.x;
  if (b < 13 * g.nz) {
    const int zi = b / 13, x = b % 13;
    const int l = x == 0 ? 0 : 1 + (x - 1) / 4, mt = x == 0 ? 0 : (x - 1) % 4;
    const int m = 32 * mt + c, n = 32 * wv + c;
    const int fan = fan_in(l);
    const bf16* A = (l == 0 ? g.XT : g.HT + (l - 1) * g.layer) + TILE * m + 8 * h;
    const bf16* B = g.DT + l * g.layer + TILE * n + 8 * h;
    const bool a_ok = m < fan;
    const int k_lo = zi * K_SPLIT, k_hi = min(g.nb, k_lo + K_SPLIT);
    f32x16 acc = {};
    for (int k0 = k_lo; k0 < k_hi; k0 += 128) {  // nb and K_SPLIT are multiples of 128
      bf16x8 av[8], bv[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int64_t k = k0 + 32 * (q >> 1);  // the tile's first row; its second sixteen for odd q
        av[q] = bf16x8{};
        if (a_ok) av[q] = *reinterpret_cast<const bf16x8*>(A + k * fan + 16 * (q & 1));
        bv[q] = *reinterpret_cast<const bf16x8*>(B + k * WD + 16 * (q & 1));
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) acc = mfma32(av[q], bv[q], acc);
    }
    float* out = g.part + (int64_t)g.nz * q_off(l) + (int64_t)zi * fan * WD;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = 32 * mt + 8 * (r >> 2) + 4 * h + (r & 3);
      if (row < fan) out[(int64_t)row * WD + n] = acc[r];
    }
    return;
  }
  b -= 13 * g.nz;
  if (b < 3 * COL_BLOCKS) {
    const int blk = b / 3, col = 256 * (b % 3) + t;
    if (col >= COLS) return;
    const int chunk = (g.nb + COL_BLOCKS - 1) / COL_BLOCKS;  // even: nb is a multiple of 128
    const int r0 = blk * chunk, r1 = min(g.nb, r0 + chunk);
    float s0 = 0.0f, s1 = 0.0f;
    const bool plain = col < NH * WD, last = col == COLS - 1;  // last: db4, the sum of dy
    const int unit = last ? 0 : col % WD;
    const bf16* x = (plain ? g.DT + (col / WD) * g.layer : g.HT + (NH - 1) * g.layer) + TILE * unit;
    if (chunk % TILE == 0) {
      // whole tiles: 64 contiguous bytes each
      for (int r = r0; r < r1; r += TILE) {
        bf16x8 v[4];
        float d[TILE];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = *reinterpret_cast<const bf16x8*>(x + (int64_t)r * WD + 8 * q);
        if (!plain) {
#pragma unroll
          for (int q = 0; q < TILE; ++q) d[q] = g.dy[r + q];
        }
#pragma unroll
        for (int q = 0; q < TILE; q += 2) {
          const float x0 = last ? 1.0f : (float)v[q >> 3][q & 7];
          const float x1 = last ? 1.0f : (float)v[q >> 3][(q & 7) + 1];
          s0 = s0 + (plain ? x0 : x0 * d[q]);
          s1 = s1 + (plain ? x1 : x1 * d[q + 1]);
        }
      }
    } else {
      for (int r = r0; r < r1; r += 2) {
        const int64_t at = (int64_t)(r & ~(TILE - 1)) * WD + (r & (TILE - 1));
        const float x0 = last ? 1.0f : (float)x[at], x1 = last ? 1.0f : (float)x[at + 1];
        s0 = s0 + (plain ? x0 : x0 * g.dy[r]);
        s1 = s1 + (plain ? x1 : x1 * g.dy[r + 1]);
      }
    }
    g.cpart[(int64_t)blk * COLS + col] = s0 + s1;
    return;
  }
  double s = 0.0;
  for (int r = t; r < g.nb; r += LOSS_PARTS) s = s + (double)g.err[r] * (double)g.err[r];
  g.lpart[t] = s;
}

// Sum of parameter p's gradient over the splits or row blocks, in order.
__device__ __forceinline__ float sum_parts(int64_t p, int nz, const float* __restrict__ part,
                                           const float* __restrict__ cpart) {
  float a = 0.0f;
  int col = -1;
#pragma unroll
  for (int l = 0; l < NH; ++l) {
    if (p >= w_off(l) && p < b_off(l)) {
      const int64_t len = (int64_t)fan_in(l) * WD;
      const float* q = part + (int64_t)nz * q_off(l) + (p - w_off(l));
      int z = 0;
      for (; z + 16 <= nz; z += 16) {  // sixteen loads in flight
        float v[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k] = q[(z + k) * len];
#pragma unroll
        for (int k = 0; k < 16; ++k) a += v[k];
      }
      for (; z < nz; ++z) a += q[z * len];
      return a;
    }
    if (p >= b_off(l) && p < b_off(l) + WD) col = l * WD + (int)(p - b_off(l));
  }
  if (col < 0) col = NH * WD + (int)(p - W4_OFF);  // w4, then b4
  float v[COL_BLOCKS];
#pragma unroll
  for (int z = 0; z < COL_BLOCKS; ++z) v[z] = cpart[(int64_t)z * COLS + col];
#pragma unroll
  for (int z = 0; z < COL_BLOCKS; ++z) a += v[z];
  return a;
}

__global__ void k_mlp_sum(int nz, const float* __restrict__ part, const float* __restrict__ cpart,
                          float* __restrict__ grad) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < NP) grad[p] = sum_parts(p, nz, part, cpart);
}

__device__ __forceinline__ void write_copies(int64_t p, float w, bf16* Wb, bf16* Wtb) {
#pragma unroll
  for (int l = 0; l < NH; ++l)
    if (p >= w_off(l) && p < b_off(l)) {
      const int64_t q = p - w_off(l);
      const int i = (int)(q / WD), o = (int)(q % WD);
      Wb[q_off(l) + q] = (bf16)w;
      Wtb[q_off(l) + (int64_t)o * fan_in(l) + i] = (bf16)w;
    }
}

__global__ void k_refresh(const float* __restrict__ prm, bf16* Wb, bf16* Wtb) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < NP) write_copies(p, prm[p], Wb, Wtb);
}

// Adam with bias corrections c1 = 1 / (1 - beta1^t), c2 = 1 / (1 - beta2^t).
struct adam_args {
  float *prm, *m, *v;
  float lr, b1, b2, eps, c1, c2;
  bf16 *Wb, *Wtb;
};

__device__ __forceinline__ void adam_update(const adam_args& o, int64_t p, float g) {
  const float mm = o.b1 * o.m[p] + (1.0f - o.b1) * g;
  const float vv = o.b2 * o.v[p] + (1.0f - o.b2) * g * g;
  o.m[p] = mm;
  o.v[p] = vv;
  const float w = o.prm[p] - o.lr * (mm * o.c1) / (sqrtf(vv * o.c2) + o.eps);
  o.prm[p] = w;
  write_copies(p, w, o.Wb, o.Wtb);
}

__global__ void k_adam(adam_args o, const float* __restrict__ grad) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < NP) adam_update(o, p, grad[p]);
}

__global__ void k_mlp_update(adam_args o, int nz, const float* __restrict__ part,
                             const float* __restrict__ cpart) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < NP) adam_update(o, p, sum_parts(p, nz, part, cpart));
}

__global__ void k_to_bf16(int64_t n, const float* __restrict__ x, bf16* y) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = (bf16)x[i];
}

// An epoch's order of the rows: the shuffle pi applied to the order before it.
__global__ void k_reorder(int64_t n, const int32_t* __restrict__ before, const int32_t* __restrict__ pi,
                          int32_t* __restrict__ after) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) after[i] = before ? before[pi[i]] : pi[i];
}

// ---------------------------------------------------------------------------------------------
// inference
// ---------------------------------------------------------------------------------------------
// Packed A fragments: element (l, ob, kb, lane, e) = W_l^T[ob*32 + lane%32][kb*16 + u(e)] with
// u = 8 h + e for layer 0 (features in natural order, h = lane / 32) and
// u = 8 (e / 4) + 4 h + e % 4 for layers 1..3.  The accumulator of a 32 x 32 MFMA holds, in lane
// (h, c) and register r, row 8 (r/4) + 4 h + r%4; registers 0..7 and 8..15 of output block ob
// are handed on unchanged as the B operands of k-blocks 2 ob and 2 ob + 1, whose slot 8 h + e
// therefore carries hidden unit 16 kb + 8 (e/4) + 4 h + e%4 -- the u above.
__global__ void k_pack(const bf16* __restrict__ Wtb, bf16* pk) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= NQ) return;
  int l = 0;
  while (l + 1 < NH && t >= q_off(l + 1)) ++l;
  const int64_t q = t - q_off(l);
  const int e = (int)(q & 7), lane = (int)((q >> 3) & 63);
  const int nkb = fan_in(l) / 16;
  const int rest = (int)(q >> 9), kb = rest % nkb, ob = rest / nkb;
  const int h = lane >> 5, r = lane & 31;
  const int u = l == 0 ? 8 * h + e : 8 * (e >> 2) + 4 * h + (e & 3);
  pk[t] = Wtb[q_off(l) + (int64_t)(ob * 32 + r) * fan_in(l) + kb * 16 + u];
}

struct infer_args {
  int64_t n;
  const double *theta, *z, *a1, *a2;
  const uint8_t* pair_cls;  // optional: class pair of entry p, ci * n_chir + cj
  int32_t n_chir;
  int32_t cls_d, cls_a;     // used without pair_cls
  int8_t cmap[16];          // context chirality id -> surrogate class
  double T;
  float tfeat, tinv;
  bool t_ok;
  const bf16* pk;
  const float* prm;
  domain_consts dom;
  const uint8_t* rmap;
  int32_t rdims[5];
  double* rate;
  uint8_t* flag;
};

constexpr int PK_VEC = (int)(NQ / 8);      // 6400 A fragments of 16 bytes
constexpr int SB_N = NH * WD + WD + 1;     // hidden biases, w4, b4

// Output block ob of a layer with its biases as the accumulator's start: element r of lane
// (h, c) of a 32 x 32 accumulator is output unit ob 32 + 8 (r / 4) + 4 h + r % 4 of entry c.
// The biases are read from LDS where each accumulator starts: an opaque copy of h keeps the
// compiler from hoisting the loads (256 values per lane) out of the tile loop.
__device__ __forceinline__ f32x16 bias_acc(const float* bias, int ob, int h) {
  asm volatile("" : "+v"(h));
  f32x16 a;
#pragma unroll
  for (int r = 0; r < 16; ++r) a[r] = bias[ob * 32 + 8 * (r >> 2) + 4 * h + (r & 3)];
  return a;
}

// SiLU of one 32 x 32 accumulator (biases included) into the B operands of k-blocks 2 ob, 2 ob + 1
__device__ __forceinline__ void to_operands(const f32x16& acc, bf16x8& lo, bf16x8& hi) {
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const bf16 s = (bf16)silu_f(acc[r]);
    if (r < 8) lo[r] = s;
    else hi[r - 8] = s;
  }
}

template <int L>
__device__ __forceinline__ void hidden_layer(const bf16x8* s_w, const float* s_b, int lane, int h,
                                             bf16x8 (&x)[8]) {
  // the fragment offsets are the same for every tile: an opaque copy per layer keeps the
  // compiler from hoisting all 128 fragment loads (512 registers) out of the tile loop
  asm volatile("" : "+v"(lane));
  bf16x8 y[8];
#pragma unroll
  for (int ob = 0; ob < 4; ++ob) {
    f32x16 acc = bias_acc(s_b + L * WD, ob, h);
#pragma unroll
    for (int kb = 0; kb < 8; ++kb) acc = mfma32(s_w[q_off(L) / 8 + (ob * 8 + kb) * 64 + lane], x[kb], acc);
    to_operands(acc, y[2 * ob], y[2 * ob + 1]);
  }
#pragma unroll
  for (int kb = 0; kb < 8; ++kb) x[kb] = y[kb];
}

// Waves per workgroup sharing one LDS copy of the weights.  The 103 KB copy allows one workgroup
// per CU, and the kernel's 168 VGPRs allow three waves per SIMD: twelve waves fill both.
constexpr int INFER_WAVES = 12;

// One wave per tile of 32 entries (the 32 columns of the MFMA tiles); the workgroup's waves
// share the LDS copy of the weights and stride over the tiles.
__global__ __launch_bounds__(64 * INFER_WAVES) void k_mlp_infer(infer_args a) {
  __shared__ bf16x8 s_w[PK_VEC];
  __shared__ float s_b[SB_N];
  {
    const bf16x8* src = reinterpret_cast<const bf16x8*>(a.pk);
    for (int i = threadIdx.x; i < PK_VEC; i += blockDim.x) s_w[i] = src[i];
    for (int i = threadIdx.x; i < NH * WD; i += blockDim.x) s_b[i] = a.prm[b_off(i / WD) + i % WD];
    for (int i = threadIdx.x; i < WD; i += blockDim.x) s_b[NH * WD + i] = a.prm[W4_OFF + i];
    if (threadIdx.x == 0) s_b[NH * WD + WD] = a.prm[B4_OFF];
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, h = lane >> 5, c = lane & 31;
  const int64_t n_tiles = (a.n + 31) / 32;
  for (int64_t tile = (int64_t)blockIdx.x * INFER_WAVES + (threadIdx.x >> 6); tile < n_tiles;
       tile += (int64_t)gridDim.x * INFER_WAVES) {
    const int64_t e = tile * 32 + c;
    const bool live = e < a.n;
    int cd = -1, ca = -1;
    float f[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (live) {
      if (a.pair_cls) {
        const int pc = a.pair_cls[e];
        cd = a.cmap[pc / a.n_chir];
        ca = a.cmap[pc % a.n_chir];
      } else {
        cd = a.cls_d;
        ca = a.cls_a;
      }
      if (h == 0) {
        double st, ct;
        sincos(a.theta[e], &st, &ct);
        f[0] = (float)ct;
        f[1] = (float)st;
        shift_features(a.z[e], a.a1[e], a.a2[e], a.dom, f + 2);
#pragma unroll
        for (int j = 0; j < NCLS; ++j) f[5 + j] = cd == j ? 1.0f : 0.0f;
      } else {
#pragma unroll
        for (int j = 0; j < NCLS; ++j) f[j] = ca == j ? 1.0f : 0.0f;
        f[3] = a.tfeat;
        f[4] = a.tinv;
      }
    }
    bf16x8 x[8];
    // layer 0: one k-block of the 16 feature slots
    {
      int wl0 = lane;
      asm volatile("" : "+v"(wl0));
      bf16x8 x0;
#pragma unroll
      for (int k = 0; k < 8; ++k) x0[k] = (bf16)f[k];
#pragma unroll
      for (int ob = 0; ob < 4; ++ob) {
        const f32x16 acc = mfma32(s_w[ob * 64 + wl0], x0, bias_acc(s_b, ob, h));
        to_operands(acc, x[2 * ob], x[2 * ob + 1]);
      }
    }
    hidden_layer<1>(s_w, s_b, lane, h, x);
    hidden_layer<2>(s_w, s_b, lane, h, x);
    // layer 3 and the output unit
    float ys = 0.0f;
    int wl = lane;
    asm volatile("" : "+v"(wl));
#pragma unroll
    for (int ob = 0; ob < 4; ++ob) {
      f32x16 acc = bias_acc(s_b + 3 * WD, ob, h);
#pragma unroll
      for (int kb = 0; kb < 8; ++kb) acc = mfma32(s_w[q_off(3) / 8 + (ob * 8 + kb) * 64 + wl], x[kb], acc);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int u = ob * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
        ys += (float)(bf16)silu_f(acc[r]) * s_b[NH * WD + u];
      }
    }
    const float yy = ys + __shfl_xor(ys, 32, 64) + s_b[NH * WD + WD];
    if (h != 0 || !live) continue;
    const double l10 = a.dom.y_shift + a.dom.y_scale * (double)yy;
    a.rate[e] = exp(l10 * 2.302585092994045684);
    if (a.flag) {
      uint8_t fl = 0;
      if (cd < 0 || ca < 0 || !a.t_ok) {
        fl = KMC_MLP_FLAG_DOMAIN;
      } else if (a.rmap) {
        const int64_t b = bin_index(a.rdims, cd, ca, a.T, a.theta[e], a.z[e], a.a1[e], a.a2[e], a.dom);
        if (a.rmap[b]) fl = KMC_MLP_FLAG_RESIDUAL;
      }
      a.flag[e] = fl;
    }
  }
}

thread_local std::string g_mlp_err;
int mfail(int code, const std::string& m) {
  g_mlp_err = m;
  return code;
}
// The runtime's own record of the error is cleared: the next call's launches would report it again.
int hip_mfail(hipError_t e, const char* who) {
  (void)hipGetLastError();
  return mfail(e == hipErrorNoDevice ? KMC_ERR_NODEVICE : KMC_ERR_HIP,
               std::string(who) + ": " + hipGetErrorString(e));
}

}  // namespace

struct kmc_mlp {
  int device = 0;
  int n_cu = 1;  // compute units of the device (grid of the inference kernel)
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  domain_consts dom{};
  float *d_prm = nullptr, *d_grad = nullptr, *d_m = nullptr, *d_v = nullptr;
  bf16 *d_wb = nullptr, *d_wtb = nullptr, *d_pk = nullptr;
  bool pk_dirty = true;
  int64_t adam_t = 0;
  uint8_t* d_rmap = nullptr;
  int32_t rdims[5] = {0, 0, 0, 0, 0};
  // training workspace for batches of up to `cap` rows
  int64_t cap = 0;
  bf16* X = nullptr;
  float* tgt = nullptr;
  bf16 *XT = nullptr, *HT = nullptr, *DT = nullptr;
  float *y = nullptr, *dy = nullptr, *err = nullptr;
  float *part = nullptr, *cpart = nullptr;
  double* lpart = nullptr;
  float* fstage = nullptr;  // FP32 staging of host feature rows
  // host-array inference staging
  int64_t geo_cap = 0;
  double* d_geo = nullptr;
  double* d_rate = nullptr;
  uint8_t* d_flag = nullptr;
};

namespace {

#define MLP_HIP(call)                                                                      \
  do {                                                                                     \
    const hipError_t e_ = (call);                                                          \
    if (e_ != hipSuccess) return hip_mfail(e_, __func__);                                  \
  } while (0)

template <typename T>
hipError_t grow(T** p, size_t n) {
  if (*p) (void)hipFree(*p);
  *p = nullptr;
  return hipMalloc((void**)p, std::max<size_t>(n, 1) * sizeof(T));
}

int64_t round_up(int64_t n, int64_t m) { return (n + m - 1) / m * m; }

int ensure_cap(kmc_mlp* m, int64_t rows) {
  rows = round_up(std::max<int64_t>(rows, 128), 128);
  if (rows <= m->cap) return KMC_OK;
  m->cap = 0;  // until all of it has grown
  MLP_HIP(grow(&m->X, rows * IN));
  MLP_HIP(grow(&m->tgt, rows));
  MLP_HIP(grow(&m->XT, rows * IN));
  MLP_HIP(grow(&m->HT, rows * WD * NH));
  MLP_HIP(grow(&m->DT, rows * WD * NH));
  MLP_HIP(grow(&m->y, rows));
  MLP_HIP(grow(&m->dy, rows));
  MLP_HIP(grow(&m->err, rows));
  MLP_HIP(grow(&m->part, round_up(rows, K_SPLIT) / K_SPLIT * NQ));
  MLP_HIP(grow(&m->fstage, rows * IN));
  m->cap = rows;
  return KMC_OK;
}

int splits(int nb) { return (nb + K_SPLIT - 1) / K_SPLIT; }

// Forward over nb rows (a multiple of 128) of X, or of the rows idx of X; with `backward` also
// the parts of the gradient and the squared error's sums in lpart.
hipError_t step(kmc_mlp* m, int nb, int n_valid, bool backward, const bf16* X, const float* tgt,
                const int32_t* idx, double* lpart) {
  hipStream_t st = m->stream;
  rows_args g{};
  g.n_valid = n_valid;
  g.idx = idx;
  g.X = X;
  g.tgt = tgt;
  g.inv_n = 1.0f / (float)std::max(n_valid, 1);
  g.Wtb = m->d_wtb;
  g.Wb = m->d_wb;
  g.prm = m->d_prm;
  g.layer = m->cap * WD;
  g.XT = m->XT;
  g.HT = m->HT;
  g.DT = m->DT;
  g.y = m->y;
  g.dy = m->dy;
  g.err = m->err;
  const dim3 grid((unsigned)(nb / TILE));
  if (!backward) {
    hipLaunchKernelGGL(k_mlp_rows<false>, grid, dim3(256), 0, st, g);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_mlp_rows<true>, grid, dim3(256), 0, st, g);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  grads_args q{};
  q.nb = nb;
  q.nz = splits(nb);
  q.layer = m->cap * WD;
  q.XT = m->XT;
  q.HT = m->HT;
  q.DT = m->DT;
  q.dy = m->dy;
  q.err = m->err;
  q.part = m->part;
  q.cpart = m->cpart;
  q.lpart = lpart;
  hipLaunchKernelGGL(k_mlp_grads, dim3((unsigned)(13 * q.nz + 3 * COL_BLOCKS + 1)), dim3(256), 0, st, q);
  return hipGetLastError();
}

constexpr unsigned PARAM_BLOCKS = (unsigned)((NP + 255) / 256);

adam_args next_adam(kmc_mlp* m, double lr, double b1, double b2, double eps) {
  ++m->adam_t;
  const double c1 = 1.0 / (1.0 - std::pow(b1, (double)m->adam_t));
  const double c2 = 1.0 / (1.0 - std::pow(b2, (double)m->adam_t));
  m->pk_dirty = true;
  return adam_args{m->d_prm,  m->d_m,      m->d_v,    (float)lr, (float)b1, (float)b2,
                   (float)eps, (float)c1, (float)c2, m->d_wb,   m->d_wtb};
}

// One epoch's Fisher-Yates shuffle as a permutation of [0, n): the n - 1 draws of the splitmix64
// stream that start after `skip` draws.
void shuffle(int64_t n, uint64_t seed, uint64_t skip, int32_t* pi) {
  constexpr uint64_t STEP = 0x9E3779B97F4A7C15ull;
  for (int64_t i = 0; i < n; ++i) pi[i] = (int32_t)i;
  uint64_t rs = (seed ^ STEP) + skip * STEP;
  for (int64_t i = n - 1; i > 0; --i) {
    uint64_t z = (rs += STEP);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    std::swap(pi[i], pi[z % (uint64_t)(i + 1)]);
  }
}

// feature rows (host FP32) -> m->X (BF16) with rows [n, nb) zero
int load_rows(kmc_mlp* m, int64_t n, int64_t nb, const float* feat, const float* targets) {
  MLP_HIP(hipMemsetAsync(m->fstage, 0, nb * IN * sizeof(float), m->stream));
  MLP_HIP(hipMemcpyAsync(m->fstage, feat, n * IN * sizeof(float), hipMemcpyHostToDevice, m->stream));
  hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)((nb * IN + 255) / 256)), dim3(256), 0, m->stream,
                     nb * IN, m->fstage, m->X);
  MLP_HIP(hipGetLastError());
  if (targets) {
    MLP_HIP(hipMemsetAsync(m->tgt, 0, nb * sizeof(float), m->stream));
    MLP_HIP(hipMemcpyAsync(m->tgt, targets, n * sizeof(float), hipMemcpyHostToDevice, m->stream));
  }
  return KMC_OK;
}

infer_args base_infer(const kmc_mlp* m, double T) {
  infer_args a{};
  a.T = T;
  a.t_ok = T >= m->dom.t_lo && T <= m->dom.t_hi;
  a.tfeat = (float)temp_feature(T, m->dom);
  a.tinv = (float)inv_temp_feature(T, m->dom);
  a.pk = m->d_pk;
  a.prm = m->d_prm;
  a.dom = m->dom;
  a.rmap = m->d_rmap;
  for (int k = 0; k < 5; ++k) a.rdims[k] = m->rdims[k];
  return a;
}

// At most one workgroup per CU, each striding over the tiles, so that every CU copies the
// weights into LDS once per launch.
hipError_t launch_infer(const infer_args& a, int n_cu, hipStream_t st) {
  if (a.n == 0) return hipSuccess;
  const int64_t tiles = (a.n + 31) / 32;
  const unsigned grid = (unsigned)std::min<int64_t>((tiles + INFER_WAVES - 1) / INFER_WAVES, n_cu);
  hipLaunchKernelGGL(k_mlp_infer, dim3(grid), dim3(64 * INFER_WAVES), 0, st, a);
  return hipGetLastError();
}

int stage_geometry(kmc_mlp* m, int64_t n, const double* th, const double* z, const double* a1,
                   const double* a2) {
  if (n > m->geo_cap) {
    m->geo_cap = 0;  // until all of it has grown
    MLP_HIP(grow(&m->d_geo, 4 * n));
    MLP_HIP(grow(&m->d_rate, n));
    MLP_HIP(grow(&m->d_flag, n));
    m->geo_cap = n;
  }
  const double* src[4] = {th, z, a1, a2};
  for (int k = 0; k < 4; ++k)
    MLP_HIP(hipMemcpyAsync(m->d_geo + k * n, src[k], n * sizeof(double), hipMemcpyHostToDevice, m->stream));
  return KMC_OK;
}

void grid_geometry(int32_t nt, const double* th, int32_t nz, const double* z, int32_t n1,
                   const double* a1, int32_t n2, const double* a2, std::vector<double>& g) {
  const int64_t n = (int64_t)nt * nz * n1 * n2;
  g.resize(4 * n);
  int64_t e = 0;
  for (int i = 0; i < nt; ++i)
    for (int j = 0; j < nz; ++j)
      for (int k = 0; k < n1; ++k)
        for (int q = 0; q < n2; ++q, ++e) {
          g[e] = th[i];
          g[n + e] = z[j];
          g[2 * n + e] = a1[k];
          g[3 * n + e] = a2[q];
        }
}

}  // namespace

namespace cntkmc {

int mlp_device(const kmc_mlp* m) { return m->device; }

int mlp_prepare(kmc_mlp* m) {
  if (!m->pk_dirty) return KMC_OK;
  MLP_HIP(hipSetDevice(m->device));
  hipLaunchKernelGGL(k_pack, dim3((unsigned)((NQ + 255) / 256)), dim3(256), 0, m->stream, m->d_wtb, m->d_pk);
  MLP_HIP(hipGetLastError());
  MLP_HIP(hipStreamSynchronize(m->stream));
  m->pk_dirty = false;
  return KMC_OK;
}

hipError_t mlp_launch_pairs(const kmc_mlp* m, int64_t n, const double* theta, const double* z,
                            const double* a1, const double* a2, const uint8_t* pair_cls,
                            int32_t n_chir, const int32_t* chir_class, double temperature,
                            double* rate, uint8_t* flag, hipStream_t st) {
  if (n_chir < 1 || n_chir > 16) return hipErrorInvalidValue;
  infer_args a = base_infer(m, temperature);
  a.n = n;
  a.theta = theta;
  a.z = z;
  a.a1 = a1;
  a.a2 = a2;
  a.pair_cls = pair_cls;
  a.n_chir = n_chir;
  for (int k = 0; k < n_chir; ++k)
    a.cmap[k] = (int8_t)(chir_class[k] >= 0 && chir_class[k] < NCLS ? chir_class[k] : -1);
  a.rate = rate;
  a.flag = flag;
  return launch_infer(a, m->n_cu, st);
}

}  // namespace cntkmc

extern "C" {

const char* kmc_mlp_last_error(void) { return g_mlp_err.c_str(); }

int kmc_mlp_create(int32_t device, const kmc_mlp_domain* dom, kmc_mlp** out) {
  if (!dom || !out) return mfail(KMC_ERR_ARG, "kmc_mlp_create: null argument");
  *out = nullptr;
  for (int k = 0; k < 3; ++k)
    if (!(dom->box_lo[k] < dom->box_hi[k])) return mfail(KMC_ERR_ARG, "kmc_mlp_create: empty box");
  if (dom->box_lo[1] != -dom->box_hi[1] || dom->box_lo[2] != -dom->box_hi[2])
    return mfail(KMC_ERR_ARG, "kmc_mlp_create: the axis-shift box must be symmetric about 0");
  if (!(dom->t_lo > 0 && dom->t_lo < dom->t_hi) || !(dom->y_scale != 0))
    return mfail(KMC_ERR_ARG, "kmc_mlp_create: bad temperature range or output scale");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
    return mfail(KMC_ERR_NODEVICE, "kmc_mlp_create: no HIP device");
  if (device < 0 || device >= ndev) return mfail(KMC_ERR_ARG, "kmc_mlp_create: bad device index");
  kmc_mlp* m = new kmc_mlp();
  m->device = device;
  for (int k = 0; k < 3; ++k) {
    m->dom.lo[k] = dom->box_lo[k];
    m->dom.hi[k] = dom->box_hi[k];
  }
  m->dom.t_lo = dom->t_lo;
  m->dom.t_hi = dom->t_hi;
  m->dom.y_shift = dom->y_shift;
  m->dom.y_scale = dom->y_scale;
  hipError_t e = hipSetDevice(device);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&m->n_cu, hipDeviceAttributeMultiprocessorCount, device);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipEventCreate(&m->ev0);
  if (e == hipSuccess) e = hipEventCreate(&m->ev1);
  if (e == hipSuccess) e = grow(&m->d_prm, NP);
  if (e == hipSuccess) e = grow(&m->d_grad, NP);
  if (e == hipSuccess) e = grow(&m->d_m, NP);
  if (e == hipSuccess) e = grow(&m->d_v, NP);
  if (e == hipSuccess) e = grow(&m->d_wb, NQ);
  if (e == hipSuccess) e = grow(&m->d_wtb, NQ);
  if (e == hipSuccess) e = grow(&m->d_pk, NQ);
  if (e == hipSuccess) e = grow(&m->cpart, (size_t)COL_BLOCKS * COLS);
  if (e == hipSuccess) e = grow(&m->lpart, LOSS_PARTS);
  for (float* b : {m->d_prm, m->d_grad, m->d_m, m->d_v})
    if (e == hipSuccess) e = hipMemsetAsync(b, 0, NP * sizeof(float), m->stream);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_refresh, dim3((unsigned)((NP + 255) / 256)), dim3(256), 0, m->stream,
                       m->d_prm, m->d_wb, m->d_wtb);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
  if (e != hipSuccess) {
    kmc_mlp_destroy(m);
    return hip_mfail(e, "kmc_mlp_create");
  }
  *out = m;
  return KMC_OK;
}

int kmc_mlp_destroy(kmc_mlp* m) {
  if (!m) return KMC_OK;
  (void)hipSetDevice(m->device);
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  void* bufs[] = {m->d_prm, m->d_grad, m->d_m,  m->d_v,  m->d_wb,    m->d_wtb, m->d_pk,
                  m->d_rmap, m->X,     m->tgt,  m->y,    m->dy,      m->err,   m->XT,
                  m->HT,    m->DT,     m->part, m->cpart, m->lpart,  m->fstage, m->d_geo,
                  m->d_rate, m->d_flag};
  for (void* b : bufs)
    if (b) (void)hipFree(b);
  if (m->ev0) (void)hipEventDestroy(m->ev0);
  if (m->ev1) (void)hipEventDestroy(m->ev1);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
  return KMC_OK;
}

int kmc_mlp_set_params(kmc_mlp* m, const float* params) {
  if (!m || !params) return mfail(KMC_ERR_ARG, "kmc_mlp_set_params: null argument");
  MLP_HIP(hipSetDevice(m->device));
  MLP_HIP(hipMemcpyAsync(m->d_prm, params, NP * sizeof(float), hipMemcpyHostToDevice, m->stream));
  MLP_HIP(hipMemsetAsync(m->d_m, 0, NP * sizeof(float), m->stream));
  MLP_HIP(hipMemsetAsync(m->d_v, 0, NP * sizeof(float), m->stream));
  hipLaunchKernelGGL(k_refresh, dim3((unsigned)((NP + 255) / 256)), dim3(256), 0, m->stream,
                     m->d_prm, m->d_wb, m->d_wtb);
  MLP_HIP(hipGetLastError());
  MLP_HIP(hipStreamSynchronize(m->stream));
  m->adam_t = 0;
  m->pk_dirty = true;
  return KMC_OK;
}

int kmc_mlp_get_params(kmc_mlp* m, float* params) {
  if (!m || !params) return mfail(KMC_ERR_ARG, "kmc_mlp_get_params: null argument");
  MLP_HIP(hipSetDevice(m->device));
  MLP_HIP(hipMemcpyAsync(params, m->d_prm, NP * sizeof(float), hipMemcpyDeviceToHost, m->stream));
  MLP_HIP(hipStreamSynchronize(m->stream));
  return KMC_OK;
}

int kmc_mlp_set_residual_map(kmc_mlp* m, const int32_t dims[5], const uint8_t* flags) {
  if (!m) return mfail(KMC_ERR_ARG, "kmc_mlp_set_residual_map: null mlp");
  MLP_HIP(hipSetDevice(m->device));
  if (m->d_rmap) (void)hipFree(m->d_rmap);
  m->d_rmap = nullptr;
  if (!flags) return KMC_OK;
  if (!dims || dims[0] != NBIN_PAIR) return mfail(KMC_ERR_ARG, "kmc_mlp_set_residual_map: dims[0] must be 9");
  int64_t len = 1;
  for (int k = 0; k < 5; ++k) {
    if (dims[k] < 1 || dims[k] > 4096) return mfail(KMC_ERR_ARG, "kmc_mlp_set_residual_map: bad dims");
    len *= dims[k];
  }
  if (len > (int64_t)1 << 26) return mfail(KMC_ERR_ARG, "kmc_mlp_set_residual_map: map too large");
  MLP_HIP(hipMalloc((void**)&m->d_rmap, len));
  MLP_HIP(hipMemcpyAsync(m->d_rmap, flags, len, hipMemcpyHostToDevice, m->stream));
  MLP_HIP(hipStreamSynchronize(m->stream));
  for (int k = 0; k < 5; ++k) m->rdims[k] = dims[k];
  return KMC_OK;
}

int kmc_mlp_features(const kmc_mlp* m, int64_t n, const double* th, const double* z, const double* a1,
                     const double* a2, const int32_t* cd, const int32_t* ca, const double* T,
                     float* f) {
  if (!m || n < 0 || (n > 0 && (!th || !z || !a1 || !a2 || !cd || !ca || !T || !f)))
    return mfail(KMC_ERR_ARG, "kmc_mlp_features: bad argument");
  for (int64_t i = 0; i < n; ++i) {
    float* r = f + i * IN;
    std::fill(r, r + IN, 0.0f);
    r[0] = (float)std::cos(th[i]);
    r[1] = (float)std::sin(th[i]);
    shift_features(z[i], a1[i], a2[i], m->dom, r + 2);
    for (int j = 0; j < NCLS; ++j) {
      r[5 + j] = cd[i] == j ? 1.0f : 0.0f;
      r[8 + j] = ca[i] == j ? 1.0f : 0.0f;
    }
    r[11] = (float)temp_feature(T[i], m->dom);
    r[12] = (float)inv_temp_feature(T[i], m->dom);
  }
  return KMC_OK;
}

int kmc_mlp_forward(kmc_mlp* m, int64_t n, const float* feat, float* y) {
  if (!m || n < 0 || (n > 0 && (!feat || !y))) return mfail(KMC_ERR_ARG, "kmc_mlp_forward: bad argument");
  MLP_HIP(hipSetDevice(m->device));
  constexpr int64_t CH = 65536;
  for (int64_t s = 0; s < n; s += CH) {
    const int64_t k = std::min(CH, n - s), nb = round_up(k, 128);
    int st = ensure_cap(m, nb);
    if (st == KMC_OK) st = load_rows(m, k, nb, feat + s * IN, nullptr);
    if (st != KMC_OK) return st;
    MLP_HIP(step(m, (int)nb, (int)k, false, m->X, nullptr, nullptr, nullptr));
    MLP_HIP(hipMemcpyAsync(y + s, m->y, k * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    MLP_HIP(hipStreamSynchronize(m->stream));
  }
  return KMC_OK;
}

int kmc_mlp_loss_grad(kmc_mlp* m, int64_t n, const float* feat, const float* targets, double* loss,
                      float* grad) {
  if (!m || n < 1 || n > (1 << 24) || !feat || !targets)
    return mfail(KMC_ERR_ARG, "kmc_mlp_loss_grad: bad argument");
  MLP_HIP(hipSetDevice(m->device));
  const int64_t nb = round_up(n, 128);
  int st = ensure_cap(m, nb);
  if (st == KMC_OK) st = load_rows(m, n, nb, feat, targets);
  if (st != KMC_OK) return st;
  MLP_HIP(step(m, (int)nb, (int)n, true, m->X, m->tgt, nullptr, m->lpart));
  hipLaunchKernelGGL(k_mlp_sum, dim3(PARAM_BLOCKS), dim3(256), 0, m->stream, splits((int)nb), m->part,
                     m->cpart, m->d_grad);
  MLP_HIP(hipGetLastError());
  std::vector<double> lp(LOSS_PARTS);
  MLP_HIP(hipMemcpyAsync(lp.data(), m->lpart, LOSS_PARTS * sizeof(double), hipMemcpyDeviceToHost, m->stream));
  if (grad) MLP_HIP(hipMemcpyAsync(grad, m->d_grad, NP * sizeof(float), hipMemcpyDeviceToHost, m->stream));
  MLP_HIP(hipStreamSynchronize(m->stream));
  if (loss) {
    double s = 0;
    for (double v : lp) s += v;
    *loss = s / (double)n;
  }
  return KMC_OK;
}

int kmc_mlp_adam_step(kmc_mlp* m, const float* grad, double lr, double b1, double b2, double eps,
                      int64_t step_no) {
  if (!m || !grad || step_no < 1) return mfail(KMC_ERR_ARG, "kmc_mlp_adam_step: bad argument");
  MLP_HIP(hipSetDevice(m->device));
  MLP_HIP(hipMemcpyAsync(m->d_grad, grad, NP * sizeof(float), hipMemcpyHostToDevice, m->stream));
  m->adam_t = step_no - 1;
  hipLaunchKernelGGL(k_adam, dim3(PARAM_BLOCKS), dim3(256), 0, m->stream, next_adam(m, lr, b1, b2, eps),
                     m->d_grad);
  MLP_HIP(hipGetLastError());
  MLP_HIP(hipStreamSynchronize(m->stream));
  return KMC_OK;
}

int kmc_mlp_train(kmc_mlp* m, int64_t n, const float* feat, const float* targets, int32_t epochs,
                  int32_t batch, double lr, double lr_min, uint64_t seed, double* epoch_loss,
                  double* elapsed_ms) {
  if (!m || !feat || !targets || epochs < 1 || batch < 128 || batch % 128 || n < batch ||
      n > ((int64_t)1 << 30) || !(lr > 0) || lr_min < 0)
    return mfail(KMC_ERR_ARG, "kmc_mlp_train: bad argument (batch a multiple of 128, n >= batch)");
  const auto t0 = std::chrono::steady_clock::now();
  MLP_HIP(hipSetDevice(m->device));
  int st = ensure_cap(m, batch);
  if (st != KMC_OK) return st;
  const int64_t per_epoch = n / batch;
  const double total = (double)epochs * per_epoch;
  const size_t n_lp = (size_t)LOSS_PARTS * per_epoch;
  // The shuffles of the next epochs are drawn by threads of their own while the GPU works (an
  // epoch's draws start at a known place of the stream, and its permutation is applied to the
  // order before it on the device); at most 2^26 entries ahead.
  const int ahead = (int)std::max<int64_t>(
      1, std::min<int64_t>({(int64_t)epochs, 8, ((int64_t)1 << 26) / n,
                            (int64_t)std::thread::hardware_concurrency() / 2}));
  std::vector<std::vector<int32_t>> pis;
  std::vector<std::thread> drawing;
  try {
    drawing.resize(ahead);
    pis.assign(ahead, std::vector<int32_t>(n));
  } catch (const std::bad_alloc&) {
    return mfail(KMC_ERR_ALLOC, "kmc_mlp_train: no memory for the shuffles");
  }
  const auto draw_epoch = [&](int32_t ep) {
    int32_t* pi = pis[ep % ahead].data();
    const uint64_t skip = (uint64_t)ep * (uint64_t)(n - 1);
    try {
      drawing[ep % ahead] = std::thread([n, seed, skip, pi] { shuffle(n, seed, skip, pi); });
    } catch (const std::system_error&) {  // no thread to be had: drawn here
      shuffle(n, seed, skip, pi);
    }
  };
  // the data set on the device: BF16 rows, FP32 targets, the rows' order (two, used in turn) and
  // an epoch's shuffle; squared-error sums of two epochs, on the device and pinned
  float* d_f = nullptr;
  bf16* d_x = nullptr;
  float* d_t = nullptr;
  int32_t* d_idx = nullptr;
  double* d_lp = nullptr;
  double* h_lp = nullptr;
  hipEvent_t done[2] = {nullptr, nullptr}, uploaded = nullptr;
  hipError_t e = hipMalloc((void**)&d_f, n * IN * sizeof(float));
  if (e == hipSuccess) e = hipMalloc((void**)&d_x, n * IN * sizeof(bf16));
  if (e == hipSuccess) e = hipMalloc((void**)&d_t, n * sizeof(float));
  if (e == hipSuccess) e = hipMalloc((void**)&d_idx, 3 * n * sizeof(int32_t));
  if (e == hipSuccess) e = hipMalloc((void**)&d_lp, 2 * n_lp * sizeof(double));
  if (e == hipSuccess) e = hipHostMalloc((void**)&h_lp, 2 * n_lp * sizeof(double));
  for (hipEvent_t& ev : done)
    if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&uploaded, hipEventDisableTiming);
  if (e == hipSuccess)
    for (int32_t ep = 0; ep < ahead; ++ep) draw_epoch(ep);
  if (e == hipSuccess) e = hipMemcpyAsync(d_f, feat, n * IN * sizeof(float), hipMemcpyHostToDevice, m->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(d_t, targets, n * sizeof(float), hipMemcpyHostToDevice, m->stream);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)((n * IN + 255) / 256)), dim3(256), 0, m->stream,
                       n * IN, d_f, d_x);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
  if (d_f) (void)hipFree(d_f);
  // an epoch's mean loss, once its sums have arrived
  const auto read_loss = [&](int32_t ep) {
    const hipError_t w = hipEventSynchronize(done[ep & 1]);
    if (w != hipSuccess || !epoch_loss) return w;
    const double* lp = h_lp + (ep & 1) * n_lp;
    double s = 0;
    for (size_t k = 0; k < n_lp; ++k) s += lp[k];
    epoch_loss[ep] = s / ((double)per_epoch * batch);
    return w;
  };
  int64_t it = 0;
  for (int32_t ep = 0; ep < epochs && e == hipSuccess; ++ep) {
    if (drawing[ep % ahead].joinable()) drawing[ep % ahead].join();
    int32_t* pi = d_idx + 2 * n;
    int32_t* order = d_idx + (ep & 1) * n;
    e = hipMemcpyAsync(pi, pis[ep % ahead].data(), n * sizeof(int32_t), hipMemcpyHostToDevice, m->stream);
    if (e != hipSuccess) break;
    hipLaunchKernelGGL(k_reorder, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, m->stream, n,
                       ep > 0 ? d_idx + ((ep + 1) & 1) * n : nullptr, pi, order);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipEventRecord(uploaded, m->stream);
    if (ep >= 2 && e == hipSuccess) e = read_loss(ep - 2);  // before its buffers are used again
    double* lp = d_lp + (ep & 1) * n_lp;
    for (int64_t b = 0; b < per_epoch && e == hipSuccess; ++b, ++it) {
      e = step(m, batch, batch, true, d_x, d_t, order + b * batch, lp + b * LOSS_PARTS);
      const double rate = lr_min + 0.5 * (lr - lr_min) * (1.0 + std::cos(M_PI * (double)it / total));
      if (e != hipSuccess) break;
      hipLaunchKernelGGL(k_mlp_update, dim3(PARAM_BLOCKS), dim3(256), 0, m->stream,
                         next_adam(m, rate, 0.9, 0.999, 1e-8), splits(batch), m->part, m->cpart);
      e = hipGetLastError();
    }
    if (e == hipSuccess)
      e = hipMemcpyAsync(h_lp + (ep & 1) * n_lp, lp, n_lp * sizeof(double), hipMemcpyDeviceToHost, m->stream);
    if (e == hipSuccess) e = hipEventRecord(done[ep & 1], m->stream);
    // the epoch's shuffle has been read: its buffer takes the next one to draw
    if (ep + ahead < epochs && e == hipSuccess) {
      e = hipEventSynchronize(uploaded);
      if (e == hipSuccess) draw_epoch(ep + ahead);
    }
  }
  for (std::thread& t : drawing)
    if (t.joinable()) t.join();
  for (int32_t ep = std::max(0, epochs - 2); ep < epochs && e == hipSuccess; ++ep) e = read_loss(ep);
  (void)hipStreamSynchronize(m->stream);
  for (void* b : {(void*)d_x, (void*)d_t, (void*)d_idx, (void*)d_lp})
    if (b) (void)hipFree(b);
  if (h_lp) (void)hipHostFree(h_lp);
  for (hipEvent_t ev : {done[0], done[1], uploaded})
    if (ev) (void)hipEventDestroy(ev);
  if (e != hipSuccess) return hip_mfail(e, "kmc_mlp_train");
  if (elapsed_ms)
    *elapsed_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return KMC_OK;
}

int kmc_mlp_rates_device(kmc_mlp* m, int64_t n, const double* d_theta, const double* d_z,
                         const double* d_a1, const double* d_a2, int32_t cls_d, int32_t cls_a,
                         double T, double* d_rate, uint8_t* d_flag) {
  if (!m || n < 0 || (n > 0 && (!d_theta || !d_z || !d_a1 || !d_a2 || !d_rate)) || !(T > 0))
    return mfail(KMC_ERR_ARG, "kmc_mlp_rates_device: bad argument");
  const int s = cntkmc::mlp_prepare(m);
  if (s != KMC_OK) return s;
  infer_args a = base_infer(m, T);
  a.n = n;
  a.theta = d_theta;
  a.z = d_z;
  a.a1 = d_a1;
  a.a2 = d_a2;
  a.cls_d = cls_d >= 0 && cls_d < NCLS ? cls_d : -1;
  a.cls_a = cls_a >= 0 && cls_a < NCLS ? cls_a : -1;
  a.rate = d_rate;
  a.flag = d_flag;
  MLP_HIP(launch_infer(a, m->n_cu, m->stream));
  MLP_HIP(hipStreamSynchronize(m->stream));
  return KMC_OK;
}

int kmc_mlp_rates(kmc_mlp* m, int64_t n, const double* th, const double* z, const double* a1,
                  const double* a2, int32_t cls_d, int32_t cls_a, double T, double* rate,
                  uint8_t* flag, double* kernel_ms) {
  if (!m || n < 0 || (n > 0 && (!th || !z || !a1 || !a2 || !rate)) || !(T > 0))
    return mfail(KMC_ERR_ARG, "kmc_mlp_rates: bad argument");
  if (n == 0) return KMC_OK;
  int s = cntkmc::mlp_prepare(m);
  if (s == KMC_OK) s = stage_geometry(m, n, th, z, a1, a2);
  if (s != KMC_OK) return s;
  infer_args a = base_infer(m, T);
  a.n = n;
  a.theta = m->d_geo;
  a.z = m->d_geo + n;
  a.a1 = m->d_geo + 2 * n;
  a.a2 = m->d_geo + 3 * n;
  a.cls_d = cls_d >= 0 && cls_d < NCLS ? cls_d : -1;
  a.cls_a = cls_a >= 0 && cls_a < NCLS ? cls_a : -1;
  a.rate = m->d_rate;
  a.flag = m->d_flag;
  MLP_HIP(hipEventRecord(m->ev0, m->stream));
  MLP_HIP(launch_infer(a, m->n_cu, m->stream));
  MLP_HIP(hipEventRecord(m->ev1, m->stream));
  MLP_HIP(hipMemcpyAsync(rate, m->d_rate, n * sizeof(double), hipMemcpyDeviceToHost, m->stream));
  if (flag) MLP_HIP(hipMemcpyAsync(flag, m->d_flag, n, hipMemcpyDeviceToHost, m->stream));
  MLP_HIP(hipStreamSynchronize(m->stream));
  if (kernel_ms) {
    float ms = 0.f;
    MLP_HIP(hipEventElapsedTime(&ms, m->ev0, m->ev1));
    *kernel_ms = ms;
  }
  return KMC_OK;
}

int kmc_mlp_table(kmc_mlp* m, int32_t cls_d, int32_t cls_a, double T, kmc_transfer* fb, int32_t nt,
                  const double* th, int32_t nz, const double* z, int32_t n1, const double* a1,
                  int32_t n2, const double* a2, double* rates, int64_t* n_fallback,
                  double* elapsed_ms) {
  if (!m || nt < 1 || nz < 1 || n1 < 1 || n2 < 1 || !th || !z || !a1 || !a2 || !rates)
    return mfail(KMC_ERR_ARG, "kmc_mlp_table: bad argument");
  const auto t0 = std::chrono::steady_clock::now();
  std::vector<double> g;
  grid_geometry(nt, th, nz, z, n1, a1, n2, a2, g);
  const int64_t n = (int64_t)nt * nz * n1 * n2;
  std::vector<uint8_t> fl(n);
  int s = kmc_mlp_rates(m, n, g.data(), g.data() + n, g.data() + 2 * n, g.data() + 3 * n, cls_d,
                        cls_a, T, rates, fl.data(), nullptr);
  if (s != KMC_OK) return s;
  std::vector<double> sub;
  std::vector<int64_t> idx;
  // coaxial nodes (theta = 0, a1 = 0) serve every same-tube hop: always exact
  for (int64_t e = 0; e < n; ++e)
    if (fl[e] || (g[e] == 0.0 && g[2 * n + e] == 0.0)) idx.push_back(e);
  if (fb && !idx.empty()) {
    const int64_t k = (int64_t)idx.size();
    sub.resize(4 * k);
    for (int64_t i = 0; i < k; ++i)
      for (int q = 0; q < 4; ++q) sub[q * k + i] = g[q * n + idx[i]];
    std::vector<double> r(k);
    s = kmc_transfer_rates(fb, k, sub.data(), sub.data() + k, sub.data() + 2 * k, sub.data() + 3 * k,
                           r.data(), nullptr);
    if (s != KMC_OK) return mfail(s, std::string("kmc_mlp_table: ") + kmc_transfer_last_error());
    for (int64_t i = 0; i < k; ++i) rates[idx[i]] = r[i];
  }
  if (n_fallback) *n_fallback = fb ? (int64_t)idx.size() : 0;
  if (elapsed_ms)
    *elapsed_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return KMC_OK;
}

}  // extern "C"
