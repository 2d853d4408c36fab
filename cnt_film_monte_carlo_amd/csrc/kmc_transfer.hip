// kmc_transfer.hip -- exact first-order exciton-transfer rate (exciton_transfer::first_order,
// src/exciton_transfer/exciton_transfer.cpp:380-441) for batches of pair geometries.
//
// Host: relevant states, partition function, energy matching and the Q factors of every
// matched pair (exciton_transfer.cpp:226-304, exciton_transfer.h:167-196) collapse into one
// coefficient per pair of centre-of-mass momenta (a, b):
//     rate = sum_ab C_ab |J_ab|^2,
//     C_ab = sum_{matched (i,f) with momenta (a,b)} (2 pi / hb) (exp(-E_i/kT) / Z)
//                 |Q_if|^2 / (L_i L_f) * Lorentzian(E_i - E_f),
// since M = |Q J| / sqrt(L_i L_f) (exciton_transfer.cpp:415) and J depends on the two states only
// through their momenta.  Device: J_ab = sum_i sum_j u_a(i) v_b(j) / |R_i - R_j| over the A-site
// unit cells of both tubes (exciton_transfer.cpp:307-377), one workgroup per geometry, each donor
// atom moved into the acceptor's frame (the inverse of make_Ru_3d's shift / rotation) so that the
// acceptor atoms and their phases are read unchanged for every geometry.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/cntkmc.h"
#include "cnt_model.h"
#include "kmc_transfer.h"

using namespace cntkmc;


namespace {

constexpr int CHUNK = 16;     // acceptor momenta per group of the term limit
constexpr int GROUP_TERMS = 256;  // nonzero C_ab terms accepted within one such group
constexpr int MAXK = 8;       // nonzero |k_b| per kernel pass (their sums are held in registers)
constexpr int MAXTERMS = 512; // folded terms of one pass
constexpr int GEOM_BATCH = 65536;  // geometries per launch (one workgroup each)
// Launches of fewer geometries than this (the surrogate's exact fallback, single-geometry calls)
// give each (geometry, 64-atom donor chunk) its own workgroup, so that a few geometries still fill
// the GPU; the chunks' shares of J go through PART_CAP entries of device memory and a finishing
// kernel.
constexpr int64_t SPLIT_BELOW = 4096;
constexpr size_t PART_CAP = size_t(1) << 21;
constexpr int MAX_HALF = 8;   // pairs of acceptor cells that the cell loop is unrolled for, at most
constexpr int DONORS = 64;    // donor atoms per chunk: one per lane, the same in the four waves

struct ex_state {
  int ik_cm_idx, n;
  double energy;
  int ik_cm;
};

// get_relevant_states (exciton_transfer.cpp:226-270)
std::vector<ex_state> relevant_states(const cnt_model& c, double min_energy, double T) {
  const double thr = min_energy + std::abs(std::log(1.e-3) * phys::kb * T);
  std::vector<ex_state> out;
  for (int n = 0; n < c.nk_relev; n++)
    for (int ic = 0; ic < c.nk_cm; ic++) {
      const double e = c.ex_energy[(size_t)ic * c.nk_relev + n];
      if (e <= thr) out.push_back({ic, n, e, c.ik_cm0 + ic});
    }
  std::stable_sort(out.begin(), out.end(),
                   [](const ex_state& a, const ex_state& b) { return a.energy < b.energy; });
  return out;
}

// Q_partial of calculate_Q (exciton_transfer.cpp:276-296)
cplx q_partial(const cnt_model& c, const ex_state& s) {
  const double kx = s.ik_cm * c.dk_l.x, ky = s.ik_cm * c.dk_l.y;
  const cplx ef0 = std::exp(cplx(0., +1.) * (kx * 0.0 + ky * 0.0));
  const cplx ef1 = std::exp(cplx(0., +1.) * (kx * c.aCC.x + ky * c.aCC.y));
  cplx qp = 0;
  const cplx* psi = &c.ex_psi[((size_t)s.ik_cm_idx * c.nk_relev + s.n) * c.nk_c];
  for (int k = 0; k < c.nk_c; k++) {
    const int32_t* id = &c.ex_idx[((size_t)s.ik_cm_idx * c.nk_c + k) * 4];
    const cplx ccA = c.wf(id[1], id[0], 1, 0), ccB = c.wf(id[1], id[0], 1, 1);
    const cplx cvA = c.wf(id[3], id[2], 0, 0), cvB = c.wf(id[3], id[2], 0, 1);
    qp += psi[k] * (ccA * std::conj(cvA) * ef0 + ccB * std::conj(cvB) * ef1);
  }
  return qp;
}

// make_Ru_3d before shift and rotation (exciton_transfer.cpp:310-322): all unit cells, centred
// in y.  make_Ru_2d (exciton_transfer.cpp:341-351): the unrolled positions.
void tube_atoms(const cnt_model& c, std::vector<double>& r3, std::vector<vec2>& r2) {
  const int n = c.Nu * c.length;
  r3.assign((size_t)n * 4, 0.0);
  r2.assign(n, vec2{});
  for (int i = 0; i < c.length; i++)
    for (int a = 0; a < c.Nu; a++) {
      const int k = i * c.Nu + a;
      r3[4 * k + 0] = c.pos_u_3d[a].x + i * c.t_vec_3d.x;
      r3[4 * k + 1] = c.pos_u_3d[a].y + i * c.t_vec_3d.y;
      r3[4 * k + 2] = c.pos_u_3d[a].z + i * c.t_vec_3d.z;
      r2[k] = {c.pos_a[a].x + i * c.t_vec.x, c.pos_a[a].y + i * c.t_vec.y};
    }
  double ymax = r3[1], ymin = r3[1];
  for (int k = 0; k < n; k++) {
    ymax = std::max(ymax, r3[4 * k + 1]);
    ymin = std::min(ymin, r3[4 * k + 1]);
  }
  const double mid = (ymax + ymin) / 2.;
  for (int k = 0; k < n; k++) r3[4 * k + 1] -= mid;
}

// ---------------------------------------------------------------------------------------------
// device: one workgroup per geometry
// ---------------------------------------------------------------------------------------------
struct exact_args {
  int32_t na;                     // donor atoms
  int32_t nu;                     // acceptor atoms of one unit cell
  int32_t half, odd;              // pairs of acceptor cells at +-m about the tube's centre; 1: a
                                  // cell at the centre too
  int32_t nk;                     // nonzero |k_b| of this pass (the kernel's NK)
  int32_t n_terms;                // folded (a, b) terms of this pass
  int32_t accumulate;             // 0: out = pass sum; 1: out += pass sum
  const double4* donor;           // [na] centred positions (w unused)
  const double2* u;               // [nma][na]  exp(-i k_a . r)
  const double* rec;              // per unit-cell atom: x, y at the tube's centre, z, 0, then the
                                  // pass's NK phases exp(i k_b . r) there
  const double* cell;             // per pair of cells: their distance m from the centre in cells,
                                  // then cos and sin of each k_b's phase over it
  double period;                  // length T of a cell
  const int32_t* term_a;          // [n_terms] donor momentum slot
  const int32_t* term_b;          // [n_terms] 0: k_b = 0, else 1 + the |k_b|'s place in the pass
  const double* term_c;           // [n_terms] C_ab
  int64_t n_geom;
  const double *theta, *z, *a1, *a2;
  const int64_t* sel;             // optional: geometry g reads entry sel[g] and writes out[sel[g]]
  const double2* trig;            // [n_geom] (cos, sin) of geometry g's theta
  int32_t split;                  // 1: workgroup (g, blockIdx.y) does donor chunk blockIdx.y only
  double2* part;                  // split: [n_geom][chunks][n_terms] shares of J_ab
  double* out;
  double clamp_lo[3], clamp_hi[3];  // z, a1, a2 box
};

// 1/sqrt(x): the hardware estimate y (relative error about 2^-23) and one third-order step of the
// binomial series, 1/sqrt(x) = y (1 - e)^(-1/2) = y (1 + e/2 + 3 e^2/8 + ...) with e = 1 - x y^2;
// the dropped 5 e^3/16 term is below 2^-60, so the result is within rounding of FP64 (5 VALU
// operations where two Newton steps take 7).
__device__ __forceinline__ double rsqrt_f64(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

// rate = sum over terms of C_ab |J_ab|^2 (thread t holds the J of terms t and t + 256), written or
// added to out[e] by thread 0.  Products are written as explicit FMAs here and in the J sums, so
// that every kernel that shares this arithmetic rounds it the same way.
__device__ __forceinline__ void finish_rate(const exact_args& a, int64_t e, const double (&jr)[2],
                                            const double (&ji)[2], double* s_red, int tid) {
  double part = tid < a.n_terms ? a.term_c[tid] * fma(ji[0], ji[0], jr[0] * jr[0]) : 0.0;
  if (tid + 256 < a.n_terms) part += a.term_c[tid + 256] * fma(ji[1], ji[1], jr[1] * jr[1]);
  for (int off = 32; off > 0; off >>= 1) part += __shfl_down(part, off, 64);
  if ((tid & 63) == 0) s_red[tid >> 6] = part;
  __syncthreads();
  if (tid == 0) {
    const double sum = (s_red[0] + s_red[1]) + (s_red[2] + s_red[3]);
    a.out[e] = a.accumulate ? a.out[e] + sum : sum;
  }
  __syncthreads();
}

// One step of a wave sum of several values at once: the lanes below 32 (or of the even rows of
// 16) go on with x, the others with y, each having taken the partner lane's part of its value.
template <int W>
__device__ __forceinline__ double fold_pair(double x, double y) {
  const auto swap = [](uint32_t p, uint32_t q) {
    if constexpr (W == 32) return __builtin_amdgcn_permlane32_swap(p, q, false, false);
    else return __builtin_amdgcn_permlane16_swap(p, q, false, false);
  };
  const auto lo = swap((uint32_t)__double2loint(x), (uint32_t)__double2loint(y));
  const auto hi = swap((uint32_t)__double2hiint(x), (uint32_t)__double2hiint(y));
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

// x plus its value in another lane of the row of 16 (a DPP control word).
template <int CTRL>
__device__ __forceinline__ double add_dpp(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xF, 0xF, true);
  return x + __hiloint2double(hi, lo);
}

// The wave sums of four complex values at once, 34 VALU instructions where eight separate
// butterflies take 144.  The row r = lane / 16 ends with component r / 2 (the lanes 0..31 re,
// 32..63 im) of value (r & 1) in its lanes 0..7 and of value 2 + (r & 1) in its lanes 8..15.
__device__ __forceinline__ double wave_sum4(const double2 (&v)[4], uint32_t lane) {
  double c[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) c[k] = fold_pair<32>(v[k].x, v[k].y);
  const double p = fold_pair<16>(c[0], c[1]), q = fold_pair<16>(c[2], c[3]);
  const bool up = (lane & 8u) != 0u;
  const double keep = up ? q : p, give = up ? p : q;
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(give), 0x128, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(give), 0x128, 0xF, 0xF, true);
  double s = keep + __hiloint2double(hi, lo);  // row_ror:8
  s = add_dpp<0x141>(s);                       // row_half_mirror: lane 7 - i of the half row
  s = add_dpp<0x4E>(s);                        // quad_perm [2,3,0,1]
  return add_dpp<0xB1>(s);                     // quad_perm [1,0,3,2]
}

// One workgroup of 256 threads per geometry.  make_Ru_3d places the acceptor at
// R_j = Rz(theta) (b_j + s2 y) + z_s z and the donor at r_i + s1 y; since Rz leaves z and lengths
// alone, |R_i - R_j| = |q_i - b_j| with the donor atom taken into the acceptor's frame,
// q_i = Rz(-theta) (r_i + s1 y - z_s z) - s2 y, so the acceptor's data are the same for every
// geometry and are read with wave-uniform addresses (scalar loads).
//
// The FP64 VALU bounds the sums W_b(i) = sum_j v_b(j) / |q_i - b_j|; three properties cut them:
//  * W of -k_b is the conjugate of W of k_b (distances are real): only the |k_b| are summed.
//  * The acceptor is a unit cell repeated along y: for one of its atoms the part of the distance
//    across the tube is computed once for all cells.
//  * The cells lie in pairs at +-m about the tube's centre, where the phase of k_b is that of the
//    centre times exp(+-i k_b m): their inverse distances enter as sum and difference, with one
//    FMA each per k_b, and the centre's phase is applied once per atom.
// Per atom pair at NK = 2 (the momenta 0, +-1, +-2) that is ~16 issue slots (4 of them the
// hardware root) against 28 for the plain sum over atoms and momenta: with tubes of ten cells,
// 27,951 geometries of (8,6) -> (7,5) at 300 K take 63.3 -> 39.5 ms (the nine tables of three
// chiralities 1,416 -> 791 ms), one geometry 0.27 -> 0.036 ms.  Errors against an 80-bit evaluation
// of the same sum stay at rounding, 2e-16 to 4e-16 on average.
//
// Donor atoms go in chunks of 64, one per lane; the four waves take a quarter of the unit cell's
// atoms each and add their sums through LDS.  The chunk's share of J_ab = sum_i u_a(i) W_b(i) is
// then summed over the lanes, four terms at a time, the waves taking turns.  Split launches run
// one chunk per workgroup and leave its share in part[] for k_exact_finish, which adds the chunks
// in the same order, so both launch shapes give the same bits.
template <int NK, int HALF, bool ODD>
__global__ __launch_bounds__(256) void k_exact_rate(exact_args a, const double* __restrict__ rec,
                                                    const double* __restrict__ cell,
                                                    const int32_t* __restrict__ term_a,
                                                    const int32_t* __restrict__ term_b) {
  constexpr int S = 4 + 2 * NK;    // doubles per unit-cell atom
  constexpr int CS = 1 + 2 * NK;   // doubles per pair of cells
  constexpr int NB = 1 + 2 * NK;   // sums per donor: W_0, then (Re, Im) W_b
  __shared__ double s_w[4][NB][DONORS];
  __shared__ double2 s_j[MAXTERMS];
  __shared__ double s_red[4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const double period = a.period;
  const int c_lo = a.nu * wave / 4, c_hi = a.nu * (wave + 1) / 4;
  for (int64_t g = blockIdx.x; g < a.n_geom; g += gridDim.x) {
    const int64_t e = a.sel ? a.sel[g] : g;
    const double zs = fmin(fmax(a.z[e], a.clamp_lo[0]), a.clamp_hi[0]);
    const double s1 = fmin(fmax(a.a1[e], a.clamp_lo[1]), a.clamp_hi[1]);
    const double s2 = fmin(fmax(a.a2[e], a.clamp_lo[2]), a.clamp_hi[2]);
    const double cth = a.trig[g].x, sth = a.trig[g].y;
    double jr[2] = {0.0, 0.0}, ji[2] = {0.0, 0.0};
    const int i_lo = a.split ? DONORS * (int)blockIdx.y : 0;
    const int i_hi = a.split ? min(a.na, i_lo + DONORS) : a.na;
    for (int i0 = i_lo; i0 < i_hi; i0 += DONORS) {
      const int i = i0 + lane;
      const bool live = i < a.na;
      const double4 ri = live ? a.donor[i] : make_double4(0, 0, 0, 0);
      const double ry = ri.y + s1;
      const double qx = cth * ri.x + sth * ry;
      const double qy = cth * ry - sth * ri.x - s2;
      const double qz = ri.z - zs;
      double w[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) w[b] = 0.0;
      const double* at = rec + (size_t)c_lo * S;
      for (int c = c_lo; c < c_hi; ++c, at += S) {
        const double dx = qx - at[0], dy = qy - at[1], dz = qz - at[2];
        const double across = fma(dz, dz, dx * dx);
        double z0 = 0.0, cs[NK > 0 ? NK : 1], sn[NK > 0 ? NK : 1];
#pragma unroll
        for (int b = 0; b < NK; ++b) cs[b] = sn[b] = 0.0;
        const auto pair_of_cells = [&](const double* t) {
          // one rounding each (m T as a number of its own would move a whole cell by its rounding)
          const double yp = fma(-t[0], period, dy), ym = fma(t[0], period, dy);
          const double rp = rsqrt_f64(fma(yp, yp, across)), rm = rsqrt_f64(fma(ym, ym, across));
          const double sum = rp + rm, dif = rp - rm;
          z0 += sum;
#pragma unroll
          for (int b = 0; b < NK; ++b) {
            cs[b] = fma(t[1 + 2 * b], sum, cs[b]);
            sn[b] = fma(t[2 + 2 * b], dif, sn[b]);
          }
        };
        if constexpr (HALF > 0) {
          // read again for every atom (scalar loads that hit the cache) where the table, kept over
          // the loop, would spill from scalar to vector registers
          int t = 0;
          if constexpr (HALF * CS > 25) asm volatile("" : "+s"(t));
#pragma unroll
          for (int p = 0; p < HALF; ++p) pair_of_cells(cell + t + p * CS);
        } else {
          for (int p = 0; p < a.half; ++p) pair_of_cells(cell + p * CS);
        }
        if (HALF > 0 ? ODD : a.odd != 0) {
          const double r = rsqrt_f64(fma(dy, dy, across));
          z0 += r;
#pragma unroll
          for (int b = 0; b < NK; ++b) cs[b] += r;
        }
        w[0] += z0;
#pragma unroll
        for (int b = 0; b < NK; ++b) {
          const double pr = at[4 + 2 * b], pi = at[5 + 2 * b];
          w[1 + 2 * b] = fma(pr, cs[b], fma(-pi, sn[b], w[1 + 2 * b]));
          w[2 + 2 * b] = fma(pr, sn[b], fma(pi, cs[b], w[2 + 2 * b]));
        }
      }
#pragma unroll
      for (int b = 0; b < NB; ++b) s_w[wave][b][lane] = live ? w[b] : 0.0;
      __syncthreads();
      for (int k = tid; k < NB * DONORS; k += 256) {
        double* p = &s_w[0][0][0] + k;
        p[0] = (p[0] + p[NB * DONORS]) + (p[2 * NB * DONORS] + p[3 * NB * DONORS]);
      }
      __syncthreads();
      for (int t0 = 4 * wave; t0 < a.n_terms; t0 += 16) {
        double2 v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int t = t0 + k;
          v[k] = make_double2(0.0, 0.0);
          if (t < a.n_terms && live) {
            const double2 u = a.u[(size_t)term_a[t] * a.na + i];
            const int b = term_b[t];
            const double wr = s_w[0][b == 0 ? 0 : 2 * b - 1][lane];
            const double wi = b == 0 ? 0.0 : s_w[0][2 * b][lane];
            v[k] = make_double2(fma(u.x, wr, -(u.y * wi)), fma(u.x, wi, u.y * wr));
          }
        }
        const double s = wave_sum4(v, (uint32_t)lane);
        const int t = t0 + ((lane >> 4) & 1) + 2 * ((lane >> 3) & 1);
        if ((lane & 7) == 0 && t < a.n_terms)
          reinterpret_cast<double*>(&s_j[t])[lane >> 5] = s;
      }
      __syncthreads();
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int t = tid + 256 * h;
        if (t < a.n_terms) {
          if (a.split) {
            a.part[((size_t)g * gridDim.y + blockIdx.y) * a.n_terms + t] = s_j[t];
          } else {
            jr[h] += s_j[t].x;
            ji[h] += s_j[t].y;
          }
        }
      }
    }
    if (!a.split) finish_rate(a, e, jr, ji, s_red, tid);
  }
}

// Split launches: J_ab = sum over the chunks' shares in chunk order, then the rate.
__global__ __launch_bounds__(256) void k_exact_finish(exact_args a, int n_chunks) {
  __shared__ double s_red[4];
  const int tid = threadIdx.x;
  for (int64_t g = blockIdx.x; g < a.n_geom; g += gridDim.x) {
    const int64_t e = a.sel ? a.sel[g] : g;
    double jr[2] = {0.0, 0.0}, ji[2] = {0.0, 0.0};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int t = tid + 256 * h;
      if (t < a.n_terms)
        for (int c = 0; c < n_chunks; c++) {
          const double2 p = a.part[((size_t)g * n_chunks + c) * a.n_terms + t];
          jr[h] += p.x;
          ji[h] += p.y;
        }
    }
    finish_rate(a, e, jr, ji, s_red, tid);
  }
}

int n_chunks(int32_t na) { return (na + DONORS - 1) / DONORS; }

// cos and sin of each geometry's theta, ahead of the rate passes (sincos' argument reduction would
// otherwise set the register budget, and with it the occupancy, of every rate kernel).
__global__ void k_trig(int64_t n, const int64_t* sel, const double* theta, double2* trig) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n) return;
  double s, c;
  sincos(theta[sel ? sel[g] : g], &s, &c);
  trig[g] = make_double2(c, s);
}

// Geometries whose transfer has no matched state pair: the rate is exactly zero.
__global__ void k_zero_rates(int64_t n, const int64_t* sel, double* out) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g < n) out[sel ? sel[g] : g] = 0.0;
}

// One pass over at most MAXK nonzero |k_b| (and k_b = 0).  The kernel is made for every number of
// acceptor cells up to 2 MAX_HALF + 1, its cell loop unrolled: 6 to 16 % less time than the loop, the
// more the shorter the tube and the more momenta (8,000 geometries of (7,5) -> (9,7) at 300 K with 4,
// 9, 10 and 17 cells 6.5 -> 5.6, 39.5 -> 34.1, 51.8 -> 45.2 and 236 -> 217 ms); longer tubes, of which
// the loop is a small part, take the loop.
template <int NK, int HALF, bool ODD>
void launch_cells(const exact_args& a, dim3 g, hipStream_t st) {
  hipLaunchKernelGGL((k_exact_rate<NK, HALF, ODD>), g, dim3(256), 0, st, a, a.rec, a.cell, a.term_a,
                     a.term_b);
}

template <int NK, int HALF = 1>
void launch_width(const exact_args& a, dim3 g, hipStream_t st) {
  if constexpr (HALF <= MAX_HALF) {
    if (a.half != HALF) return launch_width<NK, HALF + 1>(a, g, st);
    return a.odd ? launch_cells<NK, HALF, true>(a, g, st) : launch_cells<NK, HALF, false>(a, g, st);
  }
  launch_cells<NK, 0, false>(a, g, st);
}

hipError_t launch_pass(const exact_args& a, hipStream_t st) {
  const unsigned grid = (unsigned)std::min<int64_t>(a.n_geom, GEOM_BATCH);
  const int chunks = n_chunks(a.na);
  const dim3 g(grid, a.split ? chunks : 1);
  switch (a.nk) {
    case 0: launch_width<0>(a, g, st); break;
    case 1: launch_width<1>(a, g, st); break;
    case 2: launch_width<2>(a, g, st); break;
    case 3: launch_width<3>(a, g, st); break;
    case 4: launch_width<4>(a, g, st); break;
    case 5: launch_width<5>(a, g, st); break;
    case 6: launch_width<6>(a, g, st); break;
    case 7: launch_width<7>(a, g, st); break;
    case 8: launch_width<8>(a, g, st); break;
    default: return hipErrorInvalidValue;
  }
  if (a.split) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_exact_finish, dim3(grid), dim3(256), 0, st, a, chunks);
  }
  return hipGetLastError();
}

thread_local std::string g_tr_err;
int tfail(int code, const std::string& m) {
  if (code == KMC_ERR_HIP) (void)hipGetLastError();  // the next call's launches would report it again
  g_tr_err = m;
  return code;
}

}  // namespace

struct kmc_transfer {
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  kmc_transfer_info info{};
  std::vector<int> mom_a, mom_b;            // ik_cm of each momentum slot
  std::vector<int32_t> term_a, term_b;      // nonzero terms
  std::vector<double> term_c;
  // a pass sums nk nonzero |k_b|; folded terms [t0, t0 + nt), records at h_rec[rec0], cells at
  // h_rec[cell0]
  struct pass { int nk, t0, nt; size_t rec0, cell0; };
  std::vector<pass> passes;
  std::vector<int32_t> fold_a, fold_b;      // the device's terms: (k_a, k_b) and (-k_a, -k_b), whose
  std::vector<double> fold_c;               // J are conjugates, are one term
  int nu = 0, length = 0;                   // acceptor: unit-cell atoms and cells
  double period = 0.0;                      // and the length of a cell
  double clamp_lo[3] = {-1e300, -1e300, -1e300}, clamp_hi[3] = {1e300, 1e300, 1e300};
  std::vector<double> h_donor;
  std::vector<vec2> r2d;
  std::vector<cplx> h_u;
  std::vector<double> h_rec;                // per pass: unit-cell atoms, then pairs of cells
  bool on_device = false;
  double4* d_donor = nullptr;
  double2* d_u = nullptr;
  double* d_rec = nullptr;
  double2* d_trig = nullptr;                // [GEOM_BATCH] (cos, sin) of the batch's geometries
  double2* d_part = nullptr;                // [PART_CAP] chunk shares of J for split launches
  int32_t *d_ta = nullptr, *d_tb = nullptr;
  double* d_tc = nullptr;
  double* d_geo = nullptr;  // scratch for host-array calls: 4 n doubles
  double* d_out = nullptr;
  size_t geo_cap = 0;
};

namespace {

template <typename T>
hipError_t put(T** d, const std::vector<T>& h) {
  hipError_t e = hipMalloc((void**)d, std::max<size_t>(1, h.size()) * sizeof(T));
  if (e == hipSuccess && !h.empty()) e = hipMemcpy(*d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice);
  return e;
}

int upload(kmc_transfer* t) {
  if (t->on_device) return KMC_OK;
  hipError_t e = hipSetDevice(t->device);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&t->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipEventCreate(&t->ev0);
  if (e == hipSuccess) e = hipEventCreate(&t->ev1);
  if (e == hipSuccess) e = put((double**)&t->d_donor, t->h_donor);
  if (e == hipSuccess) e = put((cplx**)&t->d_u, t->h_u);
  if (e == hipSuccess) e = put(&t->d_rec, t->h_rec);
  if (e == hipSuccess) e = hipMalloc((void**)&t->d_trig, GEOM_BATCH * sizeof(double2));
  if (e == hipSuccess) e = hipMalloc((void**)&t->d_part, PART_CAP * sizeof(double2));
  if (e == hipSuccess) e = put(&t->d_ta, t->fold_a);
  if (e == hipSuccess) e = put(&t->d_tb, t->fold_b);
  if (e == hipSuccess) e = put(&t->d_tc, t->fold_c);
  if (e != hipSuccess)
    return tfail(e == hipErrorNoDevice ? KMC_ERR_NODEVICE : KMC_ERR_HIP,
                 std::string("kmc_transfer: device setup failed: ") + hipGetErrorString(e));
  t->on_device = true;
  return KMC_OK;
}

exact_args args_of(const kmc_transfer* t) {
  exact_args a{};
  a.na = t->info.n_atoms_donor;
  a.nu = t->nu;
  a.half = t->length / 2;
  a.odd = t->length & 1;
  a.period = t->period;
  a.donor = t->d_donor;
  a.u = t->d_u;
  a.trig = t->d_trig;
  a.part = t->d_part;
  for (int k = 0; k < 3; k++) {
    a.clamp_lo[k] = t->clamp_lo[k];
    a.clamp_hi[k] = t->clamp_hi[k];
  }
  return a;
}

// rate = sum over passes of sum_{terms of the pass} C_ab |J_ab|^2; the passes run in order on
// one stream, the first writes and the rest add.  Geometries go in batches (GEOM_BATCH, or what
// the chunk shares of a split launch fit in PART_CAP), each with its (cos, sin) table first.
hipError_t launch_exact(const kmc_transfer* t, exact_args a, hipStream_t st) {
  if (a.n_geom == 0) return hipSuccess;
  if (t->passes.empty()) {
    const unsigned grid = (unsigned)((a.n_geom + 255) / 256);
    hipLaunchKernelGGL(k_zero_rates, dim3(grid), dim3(256), 0, st, a.n_geom, a.sel, a.out);
    return hipGetLastError();
  }
  int max_terms = 1;
  for (const auto& p : t->passes) max_terms = std::max(max_terms, p.nt);
  const size_t per_geom = (size_t)n_chunks(a.na) * max_terms;  // chunk shares per geometry
  a.split = a.n_geom < SPLIT_BELOW && per_geom <= PART_CAP;
  const int64_t batch = a.split ? std::min<int64_t>(GEOM_BATCH, (int64_t)(PART_CAP / per_geom))
                                : GEOM_BATCH;
  hipError_t e = hipSuccess;
  for (int64_t g0 = 0; g0 < a.n_geom && e == hipSuccess; g0 += batch) {
    exact_args b = a;
    b.n_geom = std::min<int64_t>(batch, a.n_geom - g0);
    if (a.sel) {
      b.sel = a.sel + g0;
    } else {
      b.theta += g0;
      b.z += g0;
      b.a1 += g0;
      b.a2 += g0;
      b.out += g0;
    }
    hipLaunchKernelGGL(k_trig, dim3((unsigned)((b.n_geom + 255) / 256)), dim3(256), 0, st, b.n_geom,
                       b.sel, b.theta, t->d_trig);
    e = hipGetLastError();
    for (size_t k = 0; k < t->passes.size() && e == hipSuccess; k++) {
      const auto& p = t->passes[k];
      b.nk = p.nk;
      b.n_terms = p.nt;
      b.accumulate = k > 0;
      b.rec = t->d_rec + p.rec0;
      b.cell = t->d_rec + p.cell0;
      b.term_a = t->d_ta + p.t0;
      b.term_b = t->d_tb + p.t0;
      b.term_c = t->d_tc + p.t0;
      e = launch_pass(b, st);
    }
  }
  return e;
}

}  // namespace

namespace cntkmc {

int transfer_launch(kmc_transfer* t, int64_t n, const double* d_theta, const double* d_z,
                    const double* d_a1, const double* d_a2, const int64_t* d_sel, double* d_rate) {
  if (!t || n < 0 || (n > 0 && (!d_theta || !d_z || !d_a1 || !d_a2 || !d_rate)))
    return tfail(KMC_ERR_ARG, "kmc_transfer_rates_device: bad argument");
  if (n == 0) return KMC_OK;
  {
    const int s = upload(t);
    if (s != KMC_OK) return s;
  }
  exact_args a = args_of(t);
  a.n_geom = n;
  a.theta = d_theta;
  a.z = d_z;
  a.a1 = d_a1;
  a.a2 = d_a2;
  a.sel = d_sel;
  a.out = d_rate;
  hipError_t e = hipSetDevice(t->device);
  if (e == hipSuccess) e = launch_exact(t, a, t->stream);
  if (e != hipSuccess) return tfail(KMC_ERR_HIP, std::string("kmc_transfer_rates: ") + hipGetErrorString(e));
  return KMC_OK;
}

int transfer_wait(kmc_transfer* t) {
  const hipError_t e = hipStreamSynchronize(t->stream);
  if (e != hipSuccess) return tfail(KMC_ERR_HIP, std::string("kmc_transfer_rates: ") + hipGetErrorString(e));
  return KMC_OK;
}

}  // namespace cntkmc

extern "C" {

const char* kmc_transfer_last_error(void) { return g_tr_err.c_str(); }

int kmc_transfer_create(int32_t device, const kmc_cnt* donor, const kmc_cnt* acceptor,
                        double temperature, double broadening, kmc_transfer** out) {
  if (!donor || !acceptor || !out || !(temperature > 0) || !(broadening > 0))
    return tfail(KMC_ERR_ARG, "kmc_transfer_create: bad argument");
  *out = nullptr;
  const cnt_model& D = donor->m;
  const cnt_model& A = acceptor->m;
  using namespace phys;
  // first_order (exciton_transfer.cpp:385-400)
  double min_energy = D.ex_energy[0];
  for (double e : D.ex_energy) min_energy = std::min(min_energy, e);
  const std::vector<ex_state> ds = relevant_states(D, min_energy, temperature);
  const std::vector<ex_state> as = relevant_states(A, min_energy, temperature);
  double Z = 0;
  for (const auto& s : ds) Z += std::exp(-s.energy / (kb * temperature));
  auto lorentzian = [&](double e) { return inv_pi * broadening / (e * e + broadening * broadening); };
  kmc_transfer* t = new kmc_transfer();
  t->device = device;
  // calculate_Q coefficient (exciton_transfer.cpp:298-300)
  const double coeff = (std::pow(q0, 2) * D.Au() * A.Au()) /
                       (16 * std::pow(pi, 3) * eps0 * D.radius * A.radius *
                        std::sqrt(D.length_in_meter() * A.length_in_meter()));
  const double LiLf = D.length_in_meter() * A.length_in_meter();
  std::vector<cplx> qd(ds.size()), qa(as.size());
  for (size_t i = 0; i < ds.size(); i++) qd[i] = q_partial(D, ds[i]);
  for (size_t f = 0; f < as.size(); f++) qa[f] = q_partial(A, as[f]);
  auto slot = [](std::vector<int>& v, int k) {
    for (size_t i = 0; i < v.size(); i++)
      if (v[i] == k) return (int)i;
    v.push_back(k);
    return (int)v.size() - 1;
  };
  struct term { int p, q; double c; };
  std::vector<term> acc;  // coefficients per momentum pair, in first-match order
  int n_pairs = 0;
  // match_states (exciton_transfer.h:167-196) and the sum of first_order (:411-427)
  for (size_t i = 0; i < ds.size(); i++)
    for (size_t f = 0; f < as.size(); f++) {
      const double de = ds[i].energy - as[f].energy;
      if (!(lorentzian(de) > 1.e-2 * lorentzian(0))) continue;
      ++n_pairs;
      const cplx Q = cplx(coeff) * std::conj(qd[i]) * qa[f];
      const double w = (2 * pi / hb) * (std::exp(-ds[i].energy / (kb * temperature)) / Z) *
                       std::norm(Q) / LiLf * lorentzian(de);
      const int p = slot(t->mom_a, ds[i].ik_cm), q = slot(t->mom_b, as[f].ik_cm);
      auto it = std::find_if(acc.begin(), acc.end(), [&](const term& x) { return x.p == p && x.q == q; });
      if (it == acc.end()) acc.push_back({p, q, w});
      else it->c += w;
    }
  if (t->mom_a.empty()) t->mom_a.push_back(0);
  if (t->mom_b.empty()) t->mom_b.push_back(0);
  const int nma = (int)t->mom_a.size(), nmb = (int)t->mom_b.size();
  // terms ordered by (donor slot, acceptor slot) within groups of 16 acceptor slots
  std::sort(acc.begin(), acc.end(), [](const term& x, const term& y) {
    return x.q / CHUNK != y.q / CHUNK ? x.q / CHUNK < y.q / CHUNK : x.p != y.p ? x.p < y.p : x.q < y.q;
  });
  int group = -1, in_group = 0;
  for (const term& x : acc) {
    if (x.c == 0.0) continue;
    if (x.q / CHUNK != group) {
      group = x.q / CHUNK;
      in_group = 0;
    }
    if (++in_group > GROUP_TERMS) {
      delete t;
      return tfail(KMC_ERR_CAPACITY, "kmc_transfer_create: more than 256 momentum terms "
                                     "within 16 acceptor momenta");
    }
    t->term_a.push_back(x.p);
    t->term_b.push_back(x.q);
    t->term_c.push_back(x.c);
  }
  kmc_transfer_info& in = t->info;
  in.n_donor_states = (int)ds.size();
  in.n_acceptor_states = (int)as.size();
  in.n_pairs = n_pairs;
  in.n_mom_donor = nma;
  in.n_mom_acceptor = nmb;
  in.n_terms = (int)t->term_c.size();
  in.n_atoms_donor = D.Nu * D.length;
  in.n_atoms_acceptor = A.Nu * A.length;
  in.partition_Z = Z;
  in.min_energy = min_energy;
  // host copies of the device data; uploaded on the first rate call
  tube_atoms(D, t->h_donor, t->r2d);
  t->nu = A.Nu;
  t->length = A.length;
  t->period = A.t_vec_3d.y;
  const size_t na = t->r2d.size();
  // fold the terms: J of (-k_a, -k_b) is the conjugate of J of (k_a, k_b), so k_b >= 0 (and
  // k_a >= 0 where k_b = 0) stands for both
  struct folded { int ka, kb; double c; };
  std::vector<folded> fold;
  for (size_t k = 0; k < t->term_c.size(); k++) {
    int ka = t->mom_a[t->term_a[k]], kb = t->mom_b[t->term_b[k]];
    if (kb < 0 || (kb == 0 && ka < 0)) {
      ka = -ka;
      kb = -kb;
    }
    auto it = std::find_if(fold.begin(), fold.end(),
                           [&](const folded& x) { return x.ka == ka && x.kb == kb; });
    if (it == fold.end()) fold.push_back({ka, kb, t->term_c[k]});
    else it->c += t->term_c[k];
  }
  std::sort(fold.begin(), fold.end(), [](const folded& x, const folded& y) {
    return x.kb != y.kb ? x.kb < y.kb : x.ka < y.ka;
  });
  // passes of at most MAXK nonzero |k_b| (k_b = 0 goes with the first)
  std::vector<int> ka_slots;
  size_t next = 0;
  while (next < fold.size()) {
    kmc_transfer::pass p{0, (int)t->fold_c.size(), 0, 0, 0};
    std::vector<int> ks;
    for (; next < fold.size() && p.nt < MAXTERMS; ++next) {
      const folded& x = fold[next];
      if (x.kb != 0 && (ks.empty() || ks.back() != x.kb)) {
        if ((int)ks.size() == MAXK) break;
        ks.push_back(x.kb);
      }
      t->fold_a.push_back(slot(ka_slots, x.ka));
      t->fold_b.push_back(x.kb == 0 ? 0 : (int)ks.size());
      t->fold_c.push_back(x.c);
      ++p.nt;
    }
    p.nk = (int)ks.size();
    // unit-cell atoms at the middle of the tube (make_Ru_3d centres y between its lowest and
    // highest atom: exciton_transfer.cpp:310-322), their phases exp(i k_b . r) there; in extended
    // precision, since a cell's phase is shared by all of its atoms
    typedef long double ext;
    double ymin = A.pos_u_3d[0].y, ymax = ymin;
    for (int c = 0; c < A.Nu; c++) {
      ymin = std::min(ymin, A.pos_u_3d[c].y);
      ymax = std::max(ymax, A.pos_u_3d[c].y);
    }
    const ext T = A.t_vec_3d.y, centre = (ext)0.5 * (A.length - 1);
    const ext mid = (ymax + (A.length - 1) * T + ymin) / 2;
    const auto put_phase = [&](ext arg) {
      t->h_rec.push_back((double)std::cos(arg));
      t->h_rec.push_back((double)std::sin(arg));
    };
    p.rec0 = t->h_rec.size();
    for (int c = 0; c < A.Nu; c++) {
      t->h_rec.insert(t->h_rec.end(), {A.pos_u_3d[c].x,
                                       (double)(A.pos_u_3d[c].y + centre * T - mid),
                                       A.pos_u_3d[c].z, 0.0});
      const ext rx = A.pos_a[c].x + centre * A.t_vec.x, ry = A.pos_a[c].y + centre * A.t_vec.y;
      for (int kb : ks) put_phase(kb * ((ext)A.dk_l.x * rx + (ext)A.dk_l.y * ry));
    }
    p.cell0 = t->h_rec.size();
    for (int q = 0; q < A.length / 2; q++) {
      const ext m = A.length & 1 ? q + (ext)1 : q + (ext)0.5;  // cells from the centre
      t->h_rec.push_back((double)m);
      for (int kb : ks)
        put_phase(m * kb * ((ext)A.dk_l.x * A.t_vec.x + (ext)A.dk_l.y * A.t_vec.y));
    }
    t->passes.push_back(p);
  }
  t->h_u.assign(std::max<size_t>(1, ka_slots.size()) * na, cplx(0, 0));
  for (size_t p = 0; p < ka_slots.size(); p++) {
    const double kx = ka_slots[p] * D.dk_l.x, ky = ka_slots[p] * D.dk_l.y;
    for (size_t i = 0; i < na; i++)
      t->h_u[p * na + i] = std::exp(-cplx(0, 1) * (kx * t->r2d[i].x + ky * t->r2d[i].y));
  }
  *out = t;
  return KMC_OK;
}

int kmc_transfer_destroy(kmc_transfer* t) {
  if (!t) return KMC_OK;
  if (t->on_device) {
    (void)hipSetDevice(t->device);
    if (t->stream) (void)hipStreamSynchronize(t->stream);
    void* bufs[] = {t->d_donor, t->d_u, t->d_rec, t->d_trig, t->d_part, t->d_ta, t->d_tb, t->d_tc, t->d_geo, t->d_out};
    for (void* b : bufs)
      if (b) (void)hipFree(b);
    if (t->ev0) (void)hipEventDestroy(t->ev0);
    if (t->ev1) (void)hipEventDestroy(t->ev1);
    if (t->stream) (void)hipStreamDestroy(t->stream);
  }
  delete t;
  return KMC_OK;
}

int kmc_transfer_get_info(const kmc_transfer* t, kmc_transfer_info* info) {
  if (!t || !info) return tfail(KMC_ERR_ARG, "kmc_transfer_get_info: null argument");
  *info = t->info;
  return KMC_OK;
}

int kmc_transfer_terms(const kmc_transfer* t, int32_t* ik_cm_donor, int32_t* ik_cm_acceptor,
                       double* coef) {
  if (!t) return tfail(KMC_ERR_ARG, "kmc_transfer_terms: null argument");
  for (int k = 0; k < t->info.n_terms; k++) {
    if (ik_cm_donor) ik_cm_donor[k] = t->mom_a[t->term_a[k]];
    if (ik_cm_acceptor) ik_cm_acceptor[k] = t->mom_b[t->term_b[k]];
    if (coef) coef[k] = t->term_c[k];
  }
  return KMC_OK;
}

int kmc_transfer_set_clamp(kmc_transfer* t, const double lo[3], const double hi[3]) {
  if (!t || !lo || !hi) return tfail(KMC_ERR_ARG, "kmc_transfer_set_clamp: null argument");
  for (int k = 0; k < 3; k++) {
    if (!(lo[k] <= hi[k])) return tfail(KMC_ERR_ARG, "kmc_transfer_set_clamp: lo > hi");
    t->clamp_lo[k] = lo[k];
    t->clamp_hi[k] = hi[k];
  }
  return KMC_OK;
}

int kmc_transfer_rates_device(kmc_transfer* t, int64_t n, const double* d_theta, const double* d_z,
                              const double* d_a1, const double* d_a2, const int64_t* d_sel,
                              double* d_rate) {
  const int s = transfer_launch(t, n, d_theta, d_z, d_a1, d_a2, d_sel, d_rate);
  return s == KMC_OK && n > 0 ? transfer_wait(t) : s;
}

int kmc_transfer_rates(kmc_transfer* t, int64_t n, const double* theta, const double* z,
                       const double* a1, const double* a2, double* rate, double* kernel_ms) {
  if (!t || n < 0 || (n > 0 && (!theta || !z || !a1 || !a2 || !rate)))
    return tfail(KMC_ERR_ARG, "kmc_transfer_rates: bad argument");
  if (n == 0) return KMC_OK;
  {
    const int s = upload(t);
    if (s != KMC_OK) return s;
  }
  hipError_t e = hipSetDevice(t->device);
  if (e == hipSuccess && (size_t)n > t->geo_cap) {
    if (t->d_geo) (void)hipFree(t->d_geo);
    if (t->d_out) (void)hipFree(t->d_out);
    t->d_geo = nullptr;
    t->d_out = nullptr;
    e = hipMalloc((void**)&t->d_geo, 4 * n * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void**)&t->d_out, n * sizeof(double));
    t->geo_cap = e == hipSuccess ? (size_t)n : 0;
  }
  const double* src[4] = {theta, z, a1, a2};
  for (int q = 0; q < 4 && e == hipSuccess; q++)
    e = hipMemcpyAsync(t->d_geo + q * n, src[q], n * sizeof(double), hipMemcpyHostToDevice, t->stream);
  exact_args a = args_of(t);
  a.n_geom = n;
  a.theta = t->d_geo;
  a.z = t->d_geo + n;
  a.a1 = t->d_geo + 2 * n;
  a.a2 = t->d_geo + 3 * n;
  a.sel = nullptr;
  a.out = t->d_out;
  if (e == hipSuccess) e = hipEventRecord(t->ev0, t->stream);
  if (e == hipSuccess) e = launch_exact(t, a, t->stream);
  if (e == hipSuccess) e = hipEventRecord(t->ev1, t->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(rate, t->d_out, n * sizeof(double), hipMemcpyDeviceToHost, t->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(t->stream);
  if (e == hipSuccess && kernel_ms) {
    float ms = 0.f;
    e = hipEventElapsedTime(&ms, t->ev0, t->ev1);
    *kernel_ms = ms;
  }
  if (e != hipSuccess) return tfail(KMC_ERR_HIP, std::string("kmc_transfer_rates: ") + hipGetErrorString(e));
  return KMC_OK;
}

int kmc_transfer_table(kmc_transfer* t, int32_t nt, const double* th, int32_t nz, const double* z,
                       int32_t n1, const double* a1, int32_t n2, const double* a2, double* rates,
                       double* elapsed_ms) {
  if (!t || nt < 1 || nz < 1 || n1 < 1 || n2 < 1 || !th || !z || !a1 || !a2 || !rates)
    return tfail(KMC_ERR_ARG, "kmc_transfer_table: bad argument");
  const auto t0 = std::chrono::steady_clock::now();
  // nodes in the order of create_davoody_scatt_table's loops (monte_carlo.cpp:110-122)
  const int64_t n = (int64_t)nt * nz * n1 * n2;
  std::vector<double> g(4 * n);
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
  const int s = kmc_transfer_rates(t, n, g.data(), g.data() + n, g.data() + 2 * n, g.data() + 3 * n,
                                   rates, nullptr);
  if (s != KMC_OK) return s;
  if (elapsed_ms)
    *elapsed_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return KMC_OK;
}

}  // extern "C"

