// kmc_kernels.hip -- CDNA4 (gfx950) kernels of the KMC exciton-hopping path.
//
//   (a) cell list          k_cell_assign, k_cell_scatter, k_cell_sort
//   (b) CSR out-rate table  k_count_pairs, k_list_pairs, k_pair_values, k_finish_pair_rates
//   (c) hop kernel          k_inject, k_hop
//   (d) MSD/current reduce  k_reduce_samples
// plus a three-phase exclusive scan used by (a) and (b).
//
// Exactness: every FP64 expression that decides a neighbour, a rate, a selection or a dwell
// time is evaluated with contraction off (no FMA), in the operation order of the reference
// (src/monte_carlo/scatterer.cpp, scatterer.h, particle.cpp), so the CPU oracle reproduces
// it bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <utility>

#include "kmc_internal.h"
#include "kmc_kernels.h"
#include "philox.h"

namespace cntkmc {

// =============================================================================================
// Exclusive scan: uint32 counts -> int64 offsets, out[n] = total.
// =============================================================================================
constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

__device__ __forceinline__ int64_t block_exclusive_scan(int64_t v, int64_t* lds, int64_t* total) {
  // Wave-level inclusive scan with shuffles (64-wide wavefronts), then across the 4 waves.
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int64_t x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int64_t y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  if (lane == 63) lds[wave] = x;
  __syncthreads();
  int64_t wave_off = 0, tot = 0;
  for (int w = 0; w < SCAN_THREADS / 64; ++w) {
    if (w < wave) wave_off += lds[w];
    tot += lds[w];
  }
  __syncthreads();
  *total = tot;
  return wave_off + x - v;
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_tiles(const uint32_t* __restrict__ in,
                                                             int64_t* __restrict__ out,
                                                             int64_t* __restrict__ tile_sums,
                                                             int64_t n) {
  __shared__ int64_t lds[SCAN_THREADS / 64];
  const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
  uint32_t v[SCAN_ITEMS];
  int64_t sum = 0;
#pragma unroll
  for (int i = 0; i < SCAN_ITEMS; ++i) {
    v[i] = (base + i < n) ? in[base + i] : 0u;
    sum += v[i];
  }
  int64_t total;
  int64_t run = block_exclusive_scan(sum, lds, &total);
#pragma unroll
  for (int i = 0; i < SCAN_ITEMS; ++i) {
    if (base + i < n) out[base + i] = run;
    run += v[i];
  }
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_tile_sums(int64_t* __restrict__ tile_sums,
                                                                 int64_t n_tiles,
                                                                 int64_t* __restrict__ grand_total) {
  __shared__ int64_t lds[SCAN_THREADS / 64];
  int64_t carry = 0;
  for (int64_t base = 0; base < n_tiles; base += SCAN_THREADS) {
    const int64_t i = base + threadIdx.x;
    const int64_t v = (i < n_tiles) ? tile_sums[i] : 0;
    int64_t total;
    const int64_t ex = block_exclusive_scan(v, lds, &total);
    if (i < n_tiles) tile_sums[i] = carry + ex;
    carry += total;
  }
  if (threadIdx.x == 0) *grand_total = carry;
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_add(int64_t* __restrict__ out,
                                                           const int64_t* __restrict__ tile_sums,
                                                           int64_t n) {
  const int64_t base = (int64_t)blockIdx.x * SCAN_TILE;
  const int64_t off = tile_sums[blockIdx.x];
  for (int i = threadIdx.x; i < SCAN_TILE; i += SCAN_THREADS) {
    if (base + i < n) out[base + i] += off;
  }
}

hipError_t exclusive_scan(const uint32_t* d_in, int64_t* d_out, int64_t n, int64_t* d_tmp,
                          hipStream_t st) {
  // d_out has n+1 entries; d_tmp holds n_tiles entries.
  const int64_t n_tiles = (n + SCAN_TILE - 1) / SCAN_TILE;
  if (n_tiles > 0) {
    hipLaunchKernelGGL(k_scan_tiles, dim3((unsigned)n_tiles), dim3(SCAN_THREADS), 0, st, d_in,
                       d_out, d_tmp, n);
  }
  hipLaunchKernelGGL(k_scan_tile_sums, dim3(1), dim3(SCAN_THREADS), 0, st, d_tmp, n_tiles,
                     d_out + n);
  if (n_tiles > 0) {
    hipLaunchKernelGGL(k_scan_add, dim3((unsigned)n_tiles), dim3(SCAN_THREADS), 0, st, d_out,
                       d_tmp, n);
  }
  return hipGetLastError();
}

int64_t scan_tmp_elems(int64_t n) { return (n + SCAN_TILE - 1) / SCAN_TILE + 1; }

// =============================================================================================
// (a) Cell list (create_scatterer_buckets, src/monte_carlo/monte_carlo.h:368-416)
// =============================================================================================
__global__ __launch_bounds__(256) void k_cell_assign(site_arrays s, cell_desc c,
                                                     int32_t* __restrict__ cell_of,
                                                     uint32_t* __restrict__ cell_count) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= s.n) return;
  const int ix = cell_coord(c, 0, s.px[i]);
  const int iy = cell_coord(c, 1, s.py[i]);
  const int iz = cell_coord(c, 2, s.pz[i]);
  const int64_t idx = (int64_t)ix + (int64_t)iy * c.nx + (int64_t)iz * c.nx * c.ny;
  cell_of[i] = (int32_t)idx;
  atomicAdd(&cell_count[idx], 1u);
}

__global__ __launch_bounds__(256) void k_cell_scatter(int64_t n, const int32_t* __restrict__ cell_of,
                                                      const int64_t* __restrict__ cell_start,
                                                      uint32_t* __restrict__ cell_fill,
                                                      int32_t* __restrict__ cell_sites) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int32_t c = cell_of[i];
  const uint32_t slot = atomicAdd(&cell_fill[c], 1u);
  cell_sites[cell_start[c] + slot] = (int32_t)i;
}

// Buckets hold their sites in ascending index order (the reference pushes sites in list
// order, monte_carlo.h:389-395).  Buckets are short: insertion sort per cell.
__global__ __launch_bounds__(256) void k_cell_sort(int64_t n_cells,
                                                   const int64_t* __restrict__ cell_start,
                                                   int32_t* __restrict__ cell_sites) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n_cells) return;
  const int64_t b = cell_start[c], e = cell_start[c + 1];
  for (int64_t i = b + 1; i < e; ++i) {
    const int32_t v = cell_sites[i];
    int64_t j = i - 1;
    while (j >= b && cell_sites[j] > v) {
      cell_sites[j + 1] = cell_sites[j];
      --j;
    }
    cell_sites[j + 1] = v;
  }
}

// =============================================================================================
// (b) CSR build (find_neighbors + set_max_rate, src/monte_carlo/scatterer.cpp:34-83,
//     src/monte_carlo/scatterer.h:89-93)
// =============================================================================================
// A site has 32 lanes, one per cell of its stencil (27 of them used): lane 9 a + 3 b + e visits
// the a-th, b-th, e-th valid cell along x, y, z, so that the lanes' order is the reference's
// (x-outer, y, z-inner) and a lane's neighbours follow those of the lanes before it.  A thread per
// site walked the 27 cells one after another, each a chain of dependent loads, with one lane of a
// wave at a time in the pair arithmetic (50,101 sites and 0.22 M pairs: count 54, fill 455 us; now
// count 21, list 39, values 12 us).
constexpr uint32_t STENCIL_LANES = 32;

// Calls f(j, image of j) for the neighbours of site i in the lane's cell, those inside
// (min_distance, cutoff), ascending.
template <typename F>
__device__ __forceinline__ void cell_neighbors(const site_arrays& s, const cell_desc& c,
                                               const int64_t* __restrict__ cell_start,
                                               const int32_t* __restrict__ cell_sites, int64_t i,
                                               uint32_t lane, F&& f) {
#pragma clang fp contract(off)
  const double pix = s.px[i], piy = s.py[i], piz = s.pz[i];
  const int x = stencil_cell(c, 0, cell_coord(c, 0, pix), (int)lane / 9);
  const int y = stencil_cell(c, 1, cell_coord(c, 1, piy), (int)lane / 3 % 3);
  const int z = stencil_cell(c, 2, cell_coord(c, 2, piz), (int)lane % 3);
  if (lane >= 27u || x < 0 || y < 0 || z < 0) return;
  const int64_t cell = (int64_t)x + (int64_t)y * c.nx + (int64_t)z * c.nx * c.ny;
  const int64_t beg = cell_start[cell], end = cell_start[cell + 1];
  for (int64_t q = beg; q < end; ++q) {
    const int32_t j = cell_sites[q];
    double pjx = s.px[j], pjy = s.py[j], pjz = s.pz[j];
    if (c.periodic_mask & 1) pjx = image_of(pix, pjx, c.period[0]);
    if (c.periodic_mask & 2) pjy = image_of(piy, pjy, c.period[1]);
    if (c.periodic_mask & 4) pjz = image_of(piz, pjz, c.period[2]);
    const double dist = norm3(pix - pjx, piy - pjy, piz - pjz);
    if ((dist < c.cutoff) && (dist > c.min_distance)) f(j, pjx, pjy, pjz);
  }
}

// Neighbours of the lane's cell, and of the site's cells before it (exclusive) and altogether.
__device__ __forceinline__ uint32_t stencil_count(const site_arrays& s, const cell_desc& c,
                                                  const int64_t* __restrict__ cell_start,
                                                  const int32_t* __restrict__ cell_sites, int64_t i,
                                                  uint32_t lane, uint32_t* before) {
  uint32_t count = 0;
  if (i < s.n)
    cell_neighbors(s, c, cell_start, cell_sites, i, lane,
                   [&](int32_t, double, double, double) { ++count; });
  uint32_t sum = count;
#pragma unroll
  for (int off = 1; off < (int)STENCIL_LANES; off <<= 1) {
    const uint32_t y = (uint32_t)__shfl_up((int)sum, off, (int)STENCIL_LANES);
    if (lane >= (uint32_t)off) sum += y;
  }
  *before = sum - count;
  return (uint32_t)__shfl((int)sum, (int)STENCIL_LANES - 1, (int)STENCIL_LANES);
}

__global__ __launch_bounds__(256) void k_count_pairs(int64_t i0, site_arrays s, cell_desc c,
                                                     const int64_t* __restrict__ cell_start,
                                                     const int32_t* __restrict__ cell_sites,
                                                     uint32_t* __restrict__ deg) {
  const int64_t i = i0 + ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / STENCIL_LANES;
  const uint32_t lane = threadIdx.x % STENCIL_LANES;
  uint32_t before;
  const uint32_t n = stencil_count(s, c, cell_start, cell_sites, i, lane, &before);
  if (lane == 0 && i < s.n) deg[i] = n;
}

// The pairs, row by row: target in edge[p].col, source in the bits of cum[p] (which k_pair_values
// or k_finish_pair_rates overwrite).
__global__ __launch_bounds__(256) void k_list_pairs(int64_t i0, site_arrays s, cell_desc c,
                                                    const int64_t* __restrict__ cell_start,
                                                    const int32_t* __restrict__ cell_sites,
                                                    const int64_t* __restrict__ row_ptr,
                                                    csr_arrays out) {
  const int64_t i = i0 + ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / STENCIL_LANES;
  const uint32_t lane = threadIdx.x % STENCIL_LANES;
  uint32_t before;
  const uint32_t n = stencil_count(s, c, cell_start, cell_sites, i, lane, &before);
  if (i >= s.n) return;
  const int64_t rs = row_ptr[i];
  int64_t pos = rs + before;
  cell_neighbors(s, c, cell_start, cell_sites, i, lane, [&](int32_t j, double, double, double) {
    out.edge[pos].col = (uint32_t)j | ((s.flags[j] & 2u) ? EDGE_DRAIN_BIT : 0u);
    out.cum[pos] = __longlong_as_double((long long)i);
    ++pos;
  });
  if (lane == 0) {
    site_hdr h;
    h.rs = (uint32_t)rs;
    h.n = n;
    h.gamma = 0.0;
    out.hdr[i] = h;
  }
}

// Grid axes kept in LDS while the pairs look up their nodes; longer ones are read from memory.
constexpr int GRID_LDS = 1024;

// A thread per listed pair: displacement and geometry, then in mode 0 (table) the rate from the
// nearest-node table into cum, which k_finish_pair_rates turns into the running FP64 prefix sum
// (scatterer.cpp:63, 78-80), in mode 1 (pair) the geometry for an external rate.  Within the
// search, where a few lanes of a wave hold a pair at a time, the ~600 instructions of geometry and
// lookup took 192 us for 50,101 sites and 0.22 M pairs; here, with full waves, 12 us (list 39 us).
template <int MODE>
__global__ __launch_bounds__(256) void k_pair_values(int64_t p0, int64_t nnz, site_arrays s,
                                                     cell_desc c, table_desc t, csr_arrays out,
                                                     pair_geom_arrays geo) {
#pragma clang fp contract(off)
  __shared__ double grid[MODE == 0 ? GRID_LDS : 1];
  if (MODE == 0) {
    const int len = t.n_th + t.n_z + t.n_a1 + t.n_a2;  // the axes follow one another in memory
    if (len <= GRID_LDS) {
      for (int k = threadIdx.x; k < len; k += blockDim.x) grid[k] = t.th[k];
      t.th = grid;
      t.z = t.th + t.n_th;
      t.a1 = t.z + t.n_z;
      t.a2 = t.a1 + t.n_a1;
    }
    __syncthreads();
  }
  const int64_t p = p0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nnz) return;
  const int64_t i = (int64_t)__double_as_longlong(out.cum[p]);
  edge_rec e = out.edge[p];
  const uint32_t j = e.col & EDGE_COL_MASK;
  const double pix = s.px[i], piy = s.py[i], piz = s.pz[i];
  double pjx = s.px[j], pjy = s.py[j], pjz = s.pz[j];
  if (c.periodic_mask & 1) pjx = image_of(pix, pjx, c.period[0]);
  if (c.periodic_mask & 2) pjy = image_of(piy, pjy, c.period[1]);
  if (c.periodic_mask & 4) pjz = image_of(piz, pjz, c.period[2]);
  const pair_geom g = pair_geometry(pix, piy, piz, pjx, pjy, pjz, s.ox[i], s.oy[i], s.oz[i],
                                    s.ox[j], s.oy[j], s.oz[j]);
  e.dx = (float)(pjx - pix);
  e.dy = (float)(pjy - piy);
  e.dz = (float)(pjz - piz);
  out.edge[p] = e;
  if (MODE == 0) {
    out.cum[p] = table_rate(t, s.chir[i], s.chir[j], g);
  } else {
    geo.theta[p] = g.theta;
    geo.z[p] = g.z;
    geo.a1[p] = g.a1;
    geo.a2[p] = g.a2;
  }
}

// Pairs [p0, p0 + n) as the caller's arrays hold them (col and disp optional).
__global__ __launch_bounds__(256) void k_unpack_edges(int64_t n, const edge_rec* __restrict__ edge,
                                                      int32_t* __restrict__ col,
                                                      float* __restrict__ disp) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const edge_rec e = edge[p];
  if (col) col[p] = (int32_t)(e.col & EDGE_COL_MASK);
  if (disp) {
    disp[3 * p] = e.dx;
    disp[3 * p + 1] = e.dy;
    disp[3 * p + 2] = e.dz;
  }
}

// Row starts and total rates of n sites (either optional).
__global__ __launch_bounds__(256) void k_unpack_rows(int64_t n, const site_hdr* __restrict__ hdr,
                                                     int64_t* __restrict__ row,
                                                     double* __restrict__ gamma) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const site_hdr h = hdr[i];
  if (row) row[i] = h.rs;
  if (gamma) gamma[i] = h.gamma;
}

// Three arrays of n values interleaved: out[3 k + a].
__global__ __launch_bounds__(256) void k_interleave3(int64_t n, const double* __restrict__ x,
                                                     const double* __restrict__ y,
                                                     const double* __restrict__ z,
                                                     double* __restrict__ out) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  out[3 * k] = x[k];
  out[3 * k + 1] = y[k];
  out[3 * k + 2] = z[k];
}

// Sequential FP64 inclusive prefix sum per row from per-pair rates (scatterer.cpp:78-80).
// rates may be out.cum itself.
__global__ __launch_bounds__(256) void k_finish_pair_rates(int64_t n, const double* rates,
                                                           csr_arrays out,
                                                           int32_t* __restrict__ err) {
#pragma clang fp contract(off)
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  site_hdr h = out.hdr[i];
  double cum = 0.0;
  for (uint32_t k = 0; k < h.n; ++k) {
    const double r = rates[h.rs + k];
    if (!(r >= 0.0) || isinf(r)) atomicOr(err, 1);
    cum = (k == 0) ? r : cum + r;
    out.cum[h.rs + k] = cum;
  }
  h.gamma = h.n > 0 ? cum : 0.0;
  out.hdr[i] = h;
}

// =============================================================================================
// (c) Injection and the persistent hop kernel
// =============================================================================================
// Dwell time of ff_time (scatterer.h:74-80): -(1/Gamma) * log(r / RAND_MAX), r in [1, RAND_MAX].
// A site without neighbours (the reference's set_max_rate is undefined there) or with total
// rate 0 (1/Gamma = inf in the reference, so ff_time never falls below dt) never hops again.
__device__ __forceinline__ bool trapped(uint32_t n, double gamma) { return n == 0u || !(gamma > 0.0); }

__device__ __forceinline__ double dwell_time(uint32_t n, double gamma, uint32_t r) {
#pragma clang fp contract(off)
  if (trapped(n, gamma)) return INFINITY;
  return -recip(gamma) * log_unit(div_rand_max((double)r));
}

// ---------------------------------------------------------------------------------------------
// Row blocks: the hop kernel's copy of the CSR.  Each site owns whole 128-byte lines (the L2
// line), so a hop with at most ROW_INLINE neighbours touches exactly one line.  First line, in
// 16-byte units:
//   u0      n | site | Gamma (FP64)
//   u1..u4  cum[0..8)   FP64 prefix sums; slots n-1..7 hold +inf (the last entry is Gamma,
//                       which the header carries: a count of the slots <= dice is then the
//                       selected index without a comparison against n)
//   u5, u6  tgt[0..8)   row word of the target: first line of its block | TGT_WIDE_BIT when
//                       that block has continuation lines | EDGE_DRAIN_BIT for a drain target
//   u7      x, y, z     FP32 position of the site | 0
// A site with n > ROW_INLINE continues on the next lines: cum[8..n) then tgt[8..n).  The
// displacement of a hop is the difference of the two sites' FP32 positions, so the block needs
// no per-pair payload.
// ---------------------------------------------------------------------------------------------
constexpr uint32_t ROW_INLINE = 8;

__host__ __device__ __forceinline__ uint32_t block_lines(uint32_t n) {
  const uint32_t m = n > ROW_INLINE ? n - ROW_INLINE : 0u;
  return 1u + (12u * m + 127u) / 128u;
}

// Row word of a site whose block starts at line R.
__device__ __forceinline__ uint32_t row_word(uint32_t R, uint32_t n) {
  return R | (n > ROW_INLINE ? TGT_WIDE_BIT : 0u);
}

// Placement order of the blocks: sites sorted by the Morton (Z-order) code of their cell, so that
// any contiguous range of blocks -- one XCD's share of the sorted excitons, a workgroup's rows --
// covers a compact region of the film rather than a slab.  Only the memory layout follows this
// order; the neighbour order of every row stays the reference's.
__device__ __forceinline__ uint64_t spread3(uint32_t v) {
  uint64_t x = v & 0x1FFFFFu;
  x = (x | (x << 32)) & 0x1F00000000FFFFull;
  x = (x | (x << 16)) & 0x1F0000FF0000FFull;
  x = (x | (x << 8)) & 0x100F00F00F00F00Full;
  x = (x | (x << 4)) & 0x10C30C30C30C30C3ull;
  x = (x | (x << 2)) & 0x1249249249249249ull;
  return x;
}

__global__ __launch_bounds__(256) void k_morton_keys(int64_t n, const int32_t* __restrict__ cell_of,
                                                     int32_t nx, int32_t ny,
                                                     uint64_t* __restrict__ keys,
                                                     int32_t* __restrict__ ids) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t c = cell_of[i];
  const uint32_t ix = (uint32_t)(c % nx), iy = (uint32_t)((c / nx) % ny), iz = (uint32_t)(c / ((int64_t)nx * ny));
  keys[i] = spread3(ix) | (spread3(iy) << 1) | (spread3(iz) << 2);
  ids[i] = (int32_t)i;
}

// Lines of the q-th block in placement order (order[q] = its site; identity when NULL).
__global__ __launch_bounds__(256) void k_block_sizes(int64_t n, const site_hdr* __restrict__ hdr,
                                                     const int32_t* __restrict__ order,
                                                     uint32_t* __restrict__ lines) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  lines[q] = block_lines(hdr[order ? order[q] : q].n);
}

// roff[site] = first line of its block, from the scanned line counts in placement order.
__global__ __launch_bounds__(256) void k_place_blocks(int64_t n, const int32_t* __restrict__ order,
                                                      const int64_t* __restrict__ first,
                                                      int64_t* __restrict__ roff) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q > n) return;
  if (q == n) roff[n] = first[n];
  else roff[order[q]] = first[q];
}

// Sort keys of the excitons: the first line of their current site's block.
// An exciton is idle in a launch if its next hop falls after t_max and no MSD record falls due
// before that hop (the hop kernel would only reload and store its state).  Idle excitons key
// IDLE_KEY and sort after every block line; `alive` counts the others (the hop kernel deals only
// those positions to the XCDs) and `alive_next`, the next launch's count, starts at zero.
constexpr uint32_t IDLE_KEY = 0xFFFFFFFFu;
__global__ __launch_bounds__(256) void k_exciton_keys(int64_t n, const int32_t* __restrict__ site,
                                                      const int64_t* __restrict__ roff,
                                                      idle_test it, uint32_t* __restrict__ keys,
                                                      uint32_t* __restrict__ ids,
                                                      uint32_t* __restrict__ live) {
#pragma clang fp contract(off)
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < LIVE_SLOTS) live[e * LIVE_STRIDE] = live[e * LIVE_STRIDE + 1] = 0u;
  if (e == 0 && it.alive_next) *it.alive_next = 0u;
  bool alive = false;
  if (e < n) {
    uint32_t key = (uint32_t)roff[site[e]];
    if (it.alive) {
      const double t = it.t_next[e];
      bool idle = !(t <= it.t_max);
      if (idle && it.k_rec) {  // the hop kernel's record test: t_rec = (k + 1) dt_sample < t
        const uint32_t k = it.k_rec[e];
        idle = !(k < (uint32_t)it.n_bins && (double)(k + 1u) * it.dt_sample < t);
      }
      if (idle) key = IDLE_KEY;
      alive = !idle;
    }
    keys[e] = key;
    ids[e] = (uint32_t)e;
  }
  if (it.alive) {
    const uint64_t b = __ballot(alive);
    if ((threadIdx.x & 63u) == 0u && b != 0ull) atomicAdd(it.alive, (uint32_t)__popcll(b));
  }
}

__global__ __launch_bounds__(256) void k_pack_rows(int64_t n, const site_hdr* __restrict__ hdr,
                                                   const double* __restrict__ cum,
                                                   const edge_rec* __restrict__ edge,
                                                   const int64_t* __restrict__ roff,
                                                   const double* __restrict__ px,
                                                   const double* __restrict__ py,
                                                   const double* __restrict__ pz,
                                                   uint4* __restrict__ blocks) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const site_hdr h = hdr[i];
  uint4* b = blocks + (size_t)ROW_UNITS * (size_t)roff[i];
  uint4 head;
  head.x = h.n;
  head.y = (uint32_t)i;
  head.z = (uint32_t)__double2loint(h.gamma);
  head.w = (uint32_t)__double2hiint(h.gamma);
  b[0] = head;
  double* c = reinterpret_cast<double*>(b + 1);
  uint32_t* t = reinterpret_cast<uint32_t*>(b + 5);
  const uint32_t m = h.n > ROW_INLINE ? h.n - ROW_INLINE : 0u;
  double* ce = reinterpret_cast<double*>(b + ROW_UNITS);
  uint32_t* te = reinterpret_cast<uint32_t*>(ce + m);
  for (uint32_t k = (h.n > 0u ? h.n - 1u : 0u); k < ROW_INLINE; ++k) c[k] = INFINITY;
  for (uint32_t k = 0; k < h.n; ++k) {
    const edge_rec e = edge[h.rs + k];
    const uint32_t j = e.col & EDGE_COL_MASK;
    const uint32_t tg = row_word((uint32_t)roff[j], hdr[j].n) | (e.col & EDGE_DRAIN_BIT);
    if (k < ROW_INLINE) {
      if (k + 1u < h.n) c[k] = cum[h.rs + k];
      t[k] = tg;
    } else {
      ce[k - ROW_INLINE] = cum[h.rs + k];
      te[k - ROW_INLINE] = tg;
    }
  }
  b[7] = make_uint4(__float_as_uint((float)px[i]), __float_as_uint((float)py[i]),
                    __float_as_uint((float)pz[i]), 0u);
}

__global__ __launch_bounds__(256) void k_gather_offsets(int64_t n, const int32_t* __restrict__ idx,
                                                        const int64_t* __restrict__ roff,
                                                        const site_hdr* __restrict__ hdr,
                                                        uint32_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[i] = row_word((uint32_t)roff[idx[i]], hdr[idx[i]].n);
}

struct row_regs {
  uint32_t n, site;
  double gamma;
  double c[8];
  uint4 t0, t1;   // tgt[0..4), tgt[4..8)
  float x, y, z;
};

// Registers of a row from the eight 16-byte units of its first line.
__device__ __forceinline__ row_regs row_from_units(const uint4& h, const uint4& q0, const uint4& q1,
                                                   const uint4& q2, const uint4& q3, const uint4& t0,
                                                   const uint4& t1, const uint4& p) {
  row_regs r;
  r.t0 = t0;
  r.t1 = t1;
  r.n = h.x;
  r.site = h.y;
  r.gamma = __hiloint2double((int)h.w, (int)h.z);
  r.c[0] = __hiloint2double((int)q0.y, (int)q0.x);
  r.c[1] = __hiloint2double((int)q0.w, (int)q0.z);
  r.c[2] = __hiloint2double((int)q1.y, (int)q1.x);
  r.c[3] = __hiloint2double((int)q1.w, (int)q1.z);
  r.c[4] = __hiloint2double((int)q2.y, (int)q2.x);
  r.c[5] = __hiloint2double((int)q2.w, (int)q2.z);
  r.c[6] = __hiloint2double((int)q3.y, (int)q3.x);
  r.c[7] = __hiloint2double((int)q3.w, (int)q3.z);
  r.x = __uint_as_float(p.x);
  r.y = __uint_as_float(p.y);
  r.z = __uint_as_float(p.z);
  return r;
}

// The eight 16-byte loads of one block's first line (row word W), issued together.
__device__ __forceinline__ row_regs load_row(const uint4* __restrict__ blocks, uint32_t W) {
  const uint4* b = blocks + (size_t)ROW_UNITS * (W & TGT_LINE_MASK);
  return row_from_units(b[0], b[1], b[2], b[3], b[4], b[5], b[6], b[7]);
}

// Wave-cooperative form of load_row: every lane of the wave (all 64 active) passes the row word
// of the row it needs; the wave brings the 64 first lines into its 8 KB of LDS with eight
// direct-to-LDS loads, each fetching eight whole lines (lane j of load k takes one 16-byte unit
// of row 8k + j/8, so eight lanes cover one line), and each lane then reads its own row.  Load
// k writes lane j's unit to LDS unit 64k + j = 8 (8k + j/8) + j%8, i.e. row r owns units
// [8r, 8r + 8); the unit a lane fetches is rotated by r (unit u of row r sits in slot (u + r) % 8)
// so that the per-lane reads of one unit fall in different banks.  Replaces eight scattered
// 16-byte gathers per lane (64 lines per instruction) by eight coalesced loads (8 lines each).
typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) void global_void_t;

// The row as the wave loop holds it: header, the eight inline cumulative rates and the site's
// position.  Its targets stay in the wave's LDS copy of the line and are read by index
// (target_lds), so they take no registers.
struct coop_row {
  uint32_t n, site;
  double gamma;
  double c[8];
  float x, y, z;
};

// Byte offsets into the row blocks are 32-bit (pack_rows refuses blocks of 4 GiB or more), so
// each load takes the blocks' base from scalar registers and one 32-bit offset per lane.
// coop_issue starts the eight direct-to-LDS loads of the wave's 64 first lines; coop_finish waits
// for them (and for any other vector memory operation of the wave) and reads the lane's row.
__device__ __forceinline__ void coop_issue(const uint4* __restrict__ blocks, uint32_t W,
                                           uint4* lds_wave, uint32_t lane) {
  const uint32_t line = W & TGT_LINE_MASK;
  const uint32_t unit = ((lane & 7u) - (lane >> 3)) & 7u;
  // the eight source lines first (eight lane exchanges in flight together), then the loads
  uint32_t L[8];
#pragma unroll
  for (uint32_t k = 0; k < 8; ++k) L[k] = (uint32_t)__shfl((int)line, (int)(8u * k + (lane >> 3)), 64);
  // earlier reads of this LDS region are complete before it is overwritten
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  const char* base = reinterpret_cast<const char*>(blocks);
#pragma unroll
  for (uint32_t k = 0; k < 8; ++k) {
    const uint32_t off = L[k] * (uint32_t)(16u * ROW_UNITS) + unit * 16u;
    __builtin_amdgcn_global_load_lds((global_void_t*)(base + off), (lds_void_t*)(lds_wave + 64u * k),
                                     16, 0, 0);
  }
}

__device__ __forceinline__ coop_row coop_finish(const uint4* lds_wave, uint32_t lane) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  const uint4* my = lds_wave + 8u * lane;
  const uint4 h = my[lane & 7u], q0 = my[(1u + lane) & 7u], q1 = my[(2u + lane) & 7u],
              q2 = my[(3u + lane) & 7u], q3 = my[(4u + lane) & 7u], p = my[(7u + lane) & 7u];
  coop_row r;
  r.n = h.x;
  r.site = h.y;
  r.gamma = __hiloint2double((int)h.w, (int)h.z);
  r.c[0] = __hiloint2double((int)q0.y, (int)q0.x);
  r.c[1] = __hiloint2double((int)q0.w, (int)q0.z);
  r.c[2] = __hiloint2double((int)q1.y, (int)q1.x);
  r.c[3] = __hiloint2double((int)q1.w, (int)q1.z);
  r.c[4] = __hiloint2double((int)q2.y, (int)q2.x);
  r.c[5] = __hiloint2double((int)q2.w, (int)q2.z);
  r.c[6] = __hiloint2double((int)q3.y, (int)q3.x);
  r.c[7] = __hiloint2double((int)q3.w, (int)q3.z);
  r.x = __uint_as_float(p.x);
  r.y = __uint_as_float(p.y);
  r.z = __uint_as_float(p.z);
  return r;
}

// Target word idx < ROW_INLINE of the lane's row from the wave's LDS copy (units 5 and 6,
// rotated by the lane as coop_issue stores them).  Valid until the next coop_issue.
__device__ __forceinline__ uint32_t target_lds(const uint4* lds_wave, uint32_t lane, uint32_t idx) {
  const uint32_t slot = (5u + (idx >> 2) + lane) & 7u;
  return reinterpret_cast<const uint32_t*>(lds_wave + 8u * lane + slot)[idx & 3u];
}

// The number of entries <= d of a non-decreasing c[0..8), in 0..8: a three-step binary search
// over registers (selects, no indexing) and one more comparison for 8.  Step one tells count >= 4,
// step two count >= base + 2 (base = 0 or 4), step three count >= base + 2 b1 + 1.
__device__ __forceinline__ uint32_t count_le8(const double* c, double d) {
  const bool b2 = c[3] <= d;
  const bool b1 = (b2 ? c[5] : c[1]) <= d;
  const bool b0 = (b2 ? (b1 ? c[6] : c[4]) : (b1 ? c[2] : c[0])) <= d;
  const uint32_t idx = (b2 ? 4u : 0u) | (b1 ? 2u : 0u) | (b0 ? 1u : 0u);
  return (idx == 7u && c[7] <= d) ? 8u : idx;
}

// Index picked by update_state's binary search (scatterer.cpp:17-30): the first entry whose
// cumulative rate exceeds dice, or n-1.  Rows are non-decreasing (rates >= 0 are enforced when
// the CSR is built), so that index equals the number of leading entries k < n-1 with
// cum[k] <= dice.  The inline slots n-1..7 hold +inf, so the count over the eight inline slots
// is that number for n <= 9 without any comparison against n; a longer row continues on its
// next line.
__device__ __forceinline__ uint32_t select_entry(const uint4* __restrict__ blocks, uint32_t W,
                                                 const double* c8, uint32_t n, double dice) {
  uint32_t idx = count_le8(c8, dice);
  if (idx == 8u && n > 9u) {
    // cum[8..16): the first 64 bytes of the continuation line, which a row with n > 9 always
    // owns, read in one batch of four 16-byte loads before any comparison; then further entries
    // one at a time
    const uint32_t lim = n - 1u;
    const uint4* cu = blocks + (size_t)ROW_UNITS * (W & TGT_LINE_MASK) + ROW_UNITS;
    const uint4 e0 = cu[0], e1 = cu[1], e2 = cu[2], e3 = cu[3];
    const double c[8] = {__hiloint2double((int)e0.y, (int)e0.x), __hiloint2double((int)e0.w, (int)e0.z),
                         __hiloint2double((int)e1.y, (int)e1.x), __hiloint2double((int)e1.w, (int)e1.z),
                         __hiloint2double((int)e2.y, (int)e2.x), __hiloint2double((int)e2.w, (int)e2.z),
                         __hiloint2double((int)e3.y, (int)e3.x), __hiloint2double((int)e3.w, (int)e3.z)};
    uint32_t k = 8;
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) k += (8u + q < lim && c[q] <= dice) ? 1u : 0u;
    if (k == 16u) {
      const double* ce = reinterpret_cast<const double*>(cu);
      while (k < lim && ce[k - 8u] <= dice) ++k;
    }
    idx = k;
  }
  return idx;
}

// Target word of a continuation entry idx >= ROW_INLINE of a row with n entries.
__device__ __forceinline__ uint32_t target_wide(const uint4* __restrict__ blocks, uint32_t W,
                                                uint32_t n, uint32_t idx) {
  const uint32_t m = n - ROW_INLINE;
  const double* ce =
      reinterpret_cast<const double*>(blocks + (size_t)ROW_UNITS * (W & TGT_LINE_MASK) + ROW_UNITS);
  return reinterpret_cast<const uint32_t*>(ce + m)[idx - ROW_INLINE];
}

// Target word of entry idx: from the registers for idx < 8, else from the continuation lines.
__device__ __forceinline__ uint32_t target_of(const uint4* __restrict__ blocks, uint32_t W,
                                              const row_regs& r, uint32_t idx) {
  if (idx >= ROW_INLINE) return target_wide(blocks, W, r.n, idx);
  const uint4 q = idx < 4u ? r.t0 : r.t1;
  const uint32_t k = idx & 3u;
  return k == 0u ? q.x : k == 1u ? q.y : k == 2u ? q.z : q.w;
}

// One coordinate of a hop's displacement: FP64 difference of the two FP32 positions (exact for
// sites this close), shifted by one period on a periodic axis when it exceeds half of it.
// `half` is half the period on a periodic axis and +inf on an open one (a kernel argument, so
// it stays in scalar registers); the period is half + half, exact.  One comparison of |d| on
// the common path; the shift itself is rare.
__device__ __forceinline__ double min_image(double d, double half) {
#pragma clang fp contract(off)
  if (__builtin_expect(fabs(d) > half, 0)) d = d > half ? d - (half + half) : d + (half + half);
  return d;
}

// Per-thread write-back cache of departure counts: four (site, count) entries in LRU order,
// flushed with one atomic add into this XCD's private copy of the count array when evicted.
struct count_cache {
  uint32_t s0 = 0xFFFFFFFFu, s1 = 0xFFFFFFFFu, s2 = 0xFFFFFFFFu, s3 = 0xFFFFFFFFu;
  uint32_t n0 = 0, n1 = 0, n2 = 0, n3 = 0;

  // Selects rather than a branch per entry: the lanes of a wave hit different entries, and a
  // branch chain would run every arm under partial masks and rotate the eight registers at
  // its merge.  The entries above the hit (all four on a miss) move down one place.
  __device__ __forceinline__ void add(uint32_t s, uint32_t* __restrict__ base) {
    const bool h0 = s == s0, h1 = s == s1, h2 = s == s2, h3 = s == s3;
    if (!(h0 || h1 || h2 || h3) && n3 != 0u) atomicAdd(base + s3, n3);  // the evicted entry
    // at most one entry holds s (entries are distinct lines; empty ones hold no line), so
    // the hit's count is a sum of independent selects
    const uint32_t c = (h0 ? n0 : 0u) + (h1 ? n1 : 0u) + (h2 ? n2 : 0u) + (h3 ? n3 : 0u) + 1u;
    const bool m1 = !h0, m2 = !(h0 || h1), m3 = !(h0 || h1 || h2);
    s3 = m3 ? s2 : s3;
    n3 = m3 ? n2 : n3;
    s2 = m2 ? s1 : s2;
    n2 = m2 ? n1 : n2;
    s1 = m1 ? s0 : s1;
    n1 = m1 ? n0 : n1;
    s0 = s;
    n0 = c;
  }
  __device__ __forceinline__ void flush(uint32_t* __restrict__ base) {
    if (n0) atomicAdd(base + s0, n0);
    if (n1) atomicAdd(base + s1, n1);
    if (n2) atomicAdd(base + s2, n2);
    if (n3) atomicAdd(base + s3, n3);
  }
};

// Hardware id of the XCD running this wave (gfx950: 8 XCDs).  Only picks which private copy
// of the count array a wave updates; correctness does not depend on it (device-scope atomics).
__device__ __forceinline__ uint32_t xcd_id() {
  return (uint32_t)__builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & (KMC_COUNT_COPIES - 1u);
}

__global__ __launch_bounds__(256) void k_inject(exciton_arrays x, const uint4* __restrict__ blocks,
                                                const uint32_t* __restrict__ src_roff,
                                                uint32_t n_src, uint64_t seed) {
#pragma clang fp contract(off)
  const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= x.n) return;
  const u32x4 w = draw4(seed, e, 0, STREAM_INIT);
  const uint4 h = blocks[(size_t)ROW_UNITS * (src_roff[r31(w.v[0]) % n_src] & TGT_LINE_MASK)];
  const uint32_t r = nonzero_draw(w.v[1], w.v[3], seed, e, 0, STREAM_INIT_REDRAW);
  x.site[e] = (int32_t)h.y;
  x.t_next[e] = 0.0 + dwell_time(h.x, __hiloint2double((int)h.w, (int)h.z), r);
  x.hops[e] = 0;
  x.dx[e] = 0.0;
  x.dy[e] = 0.0;
  x.dz[e] = 0.0;
  x.drains[e] = 0;
  x.hash[e] = (FNV_OFFSET ^ (uint64_t)h.y) * FNV_PRIME;
  x.k_rec[e] = 0;
  x.heading[e] = (uint8_t)(r31(w.v[2]) & 1u);
  x.s_off[e] = 0.0;
  x.t_last[e] = 0.0;
}

// ---------------------------------------------------------------------------------------------
// Drift along the tube (particle::fly, src/monte_carlo/particle.cpp:9-54) for v > 0.  The
// exciton sits s_off beyond its current site on the segment toward the next site along its
// heading; its displacement is kept as the displacement of the current site's position (hops
// and passed segments) plus that offset.  One flight covers the whole dwell before a hop (the
// reference cuts it into 1 fs steps; the path is the same).
// ---------------------------------------------------------------------------------------------
struct flight_state {
  uint32_t R;         // first line of the current site's block
  uint32_t site;
  float x, y, z;      // the current site's FP32 position
  double s;           // distance travelled from the current site toward the next one
  uint32_t heading;   // 1 = toward `right`
  double dx, dy, dz;  // displacement of the current site's position
  uint32_t nd;        // drains
  uint64_t hs;        // visited-site hash
};

// One step along a tube: where the segment that a flight at a site follows under a heading leads.
// 32 bytes at fly_table[2 (2 line + heading)], line the first of the site's block, the tube end's
// turn (particle.cpp:18-37) and the segment's length resolved beforehand.  A flight is a chain of
// dependent loads: with a leg its first segment needs one load, issued at the hop and in flight
// while the dwell is drawn, and each site passed one more; from the sites' links and row blocks it
// was three, a square root and a second division (500 hops of 100,003 excitons at 2e5 m/s: 2.26 ms,
// with legs 1.75; loading the next leg ahead of the comparison as well changed nothing).
struct fly_leg {
  uint32_t word;     // row word of the site it leads to | its drain bit; LINK_NONE: no links
  uint32_t site;     // that site
  uint32_t heading;  // the heading along the segment (1 = toward `right`)
  double len;        // the segment's length [m]
  float x, y, z;     // that site's FP32 position
};

__device__ __forceinline__ const uint4* leg_of(const net_view& v, uint32_t W, uint32_t heading) {
  return v.fly_table + 2u * (2u * (size_t)(W & TGT_LINE_MASK) + heading);
}

__device__ __forceinline__ fly_leg leg_from_units(const uint4& p, const uint4& q) {
  return fly_leg{p.x, p.y & ~FLY_HEADING_BIT, p.y >> 31, __hiloint2double((int)p.w, (int)p.z),
                 __uint_as_float(q.x), __uint_as_float(q.y), __uint_as_float(q.z)};
}

__device__ __forceinline__ fly_leg load_leg(const net_view& v, uint32_t W, uint32_t heading) {
  const uint4* b = leg_of(v, W, heading);
  return leg_from_units(b[0], b[1]);
}

// The table, a thread per site and heading.
__global__ __launch_bounds__(256) void k_fly_table(int64_t n, const int32_t* __restrict__ left,
                                                   const int32_t* __restrict__ right,
                                                   const uint8_t* __restrict__ flags,
                                                   const int64_t* __restrict__ roff,
                                                   const site_hdr* __restrict__ hdr,
                                                   const double* __restrict__ px,
                                                   const double* __restrict__ py,
                                                   const double* __restrict__ pz, double hx, double hy,
                                                   double hz, uint4* __restrict__ table,
                                                   int32_t* __restrict__ bad) {
#pragma clang fp contract(off)
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 2 * n) return;
  const int64_t i = t >> 1;
  const int32_t l = left[i], r = right[i];
  // the heading's next site, else, at a tube end, the other one
  const int32_t nx = (t & 1) ? (r >= 0 ? r : l) : (l >= 0 ? l : r);
  uint4 a = make_uint4(LINK_NONE, 0u, 0u, 0u), b = make_uint4(0u, 0u, 0u, 0u);
  if (nx >= 0) {
    const float x = (float)px[nx], y = (float)py[nx], z = (float)pz[nx];
    const double sx = min_image((double)x - (double)(float)px[i], hx);
    const double sy = min_image((double)y - (double)(float)py[i], hy);
    const double sz = min_image((double)z - (double)(float)pz[i], hz);
    const double len = norm3(sx, sy, sz);
    if (!(len > 0.0)) *bad = 1;  // a flight would pass sites without using time
    a = make_uint4(row_word((uint32_t)roff[nx], hdr[nx].n) | ((flags[nx] & 2u) ? EDGE_DRAIN_BIT : 0u),
                   (uint32_t)nx | (nx == r ? FLY_HEADING_BIT : 0u), (uint32_t)__double2loint(len),
                   (uint32_t)__double2hiint(len));
    b = make_uint4(__float_as_uint(x), __float_as_uint(y), __float_as_uint(z), 0u);
  }
  uint4* o = table + 2 * (2 * roff[i] + (t & 1));
  o[0] = a;
  o[1] = b;
}

// Flight of duration tau; `leg` is the one at (f.R, f.heading) and follows them.  A site reached on
// the way becomes the current site; a drain site counts a drain and re-injects on a source site
// (draw of stream STREAM_FLY_DRAIN + j for the j-th drain of this flight, hop counter h), keeping
// the displacement, and the flight goes on from there, as the reference's next 1 fs step would.
// False when the flight would pass more than FLY_MAX_PASSES sites (the state is then left where the
// bound stopped it).
__device__ __forceinline__ bool fly(const net_view& v, flight_state& f, fly_leg& leg, double tau,
                                    uint32_t e, uint64_t h) {
#pragma clang fp contract(off)
  uint32_t j = 0;
  for (uint32_t pass = 0; pass < FLY_MAX_PASSES; ++pass) {
    if (leg.word == LINK_NONE) return true;  // particle.cpp:11-12
    f.heading = leg.heading;
    const double dist = leg.len - f.s;
    const double need = dist / v.velocity;
    if (!(need < tau)) {  // stops on this segment (particle.cpp:46-49)
      f.s = f.s + v.velocity * tau;
      return true;
    }
    tau = tau - need;
    f.dx = f.dx + min_image((double)leg.x - (double)f.x, v.half_per[0]);
    f.dy = f.dy + min_image((double)leg.y - (double)f.y, v.half_per[1]);
    f.dz = f.dz + min_image((double)leg.z - (double)f.z, v.half_per[2]);
    f.s = 0.0;
    const uint32_t nx = leg.word;
    f.R = nx & ~EDGE_DRAIN_BIT;
    f.site = leg.site;
    f.x = leg.x;
    f.y = leg.y;
    f.z = leg.z;
    f.hs = (f.hs ^ ((uint64_t)f.site | (2ull << 32))) * FNV_PRIME;
    if (nx & EDGE_DRAIN_BIT) {
      ++f.nd;
      const u32x4 w = draw4(v.seed, e, h, STREAM_FLY_DRAIN + j);
      ++j;
      f.R = v.src_roff[r31(w.v[0]) % v.n_src];
      const uint4 hd = v.blocks[(size_t)ROW_UNITS * (f.R & TGT_LINE_MASK)];
      const uint4 p = v.blocks[(size_t)ROW_UNITS * (f.R & TGT_LINE_MASK) + 7];
      f.site = hd.y;
      f.x = __uint_as_float(p.x);
      f.y = __uint_as_float(p.y);
      f.z = __uint_as_float(p.z);
      f.hs = (f.hs ^ ((uint64_t)f.site | (1ull << 32))) * FNV_PRIME;
    }
    leg = load_leg(v, f.R, f.heading);
  }
  return leg.word == LINK_NONE;
}

// Position of the exciton relative to its current site: s along the segment toward the next one.
__device__ __forceinline__ void fly_offset(const net_view& v, const flight_state& f,
                                           const fly_leg& leg, double& ox, double& oy, double& oz) {
#pragma clang fp contract(off)
  ox = oy = oz = 0.0;
  if (!(f.s != 0.0)) return;
  const double q = f.s / leg.len;
  ox = min_image((double)leg.x - (double)f.x, v.half_per[0]) * q;
  oy = min_image((double)leg.y - (double)f.y, v.half_per[1]) * q;
  oz = min_image((double)leg.z - (double)f.z, v.half_per[2]) * q;
}

// Adds a wave's excitons to the counts at the end of a launch: b those that a further launch could
// move, due those with t <= t_max.
__device__ __forceinline__ void add_live(uint32_t* live, uint64_t b, uint64_t due) {
  if (b != 0ull) atomicAdd(live, (uint32_t)__popcll(b));
  if (due != b) atomicAdd(live + 1, (uint32_t)__popcll(due & ~b));
}

// The hop loop of one wave (v = 0), built around the cooperative row load: every lane takes part
// in every row load, so the loop runs until no lane of the wave can hop; a lane without an
// exciton (valid false) or whose exciton has stopped keeps loading some row.  Each iteration
// takes the row of the exciton's current site and
//   (A) selects the next hop from it (draws, dice, target) and issues the load of the next row
//       -- the target's, or the source site's after a drain -- before anything else, so the load
//       is in flight while
//   (B) the hop into this row finishes (displacement, visit hash, dwell at this site) and the
//       MSD records fall due, and
//   (C) the hop selected in (A) happens if the exciton's clock allows it (t <= t_max), else the
//       exciton stops at this site and the issued load is simply not used.
// Every exciton's arithmetic and its order are those of the oracle; only
// the selection is computed before the clock test that decides whether it is used.  A drain
// target's header and position are gathered by the lanes concerned.
// COUNT: departures from the block lines [win_base, win_base + COUNT_WINDOW_LINES) are counted
// in the workgroup's LDS window `win` (zeroed and flushed by the kernel), the rest through a
// four-entry register LRU into the XCD's copy of the counts.  The window holds 16-bit counters,
// two lines per word, so that 8 KB of LDS cover 4,096 lines.  A counter never wraps: the
// departure whose add returns 0x7FFF (taking the counter to 0x8000) subtracts 0x8000 from it
// again and adds 0x8000 to the line's device count.  Exactly one lane sees each such return,
// and its subtraction follows its add within a few iterations of the other waves, far fewer
// than the 0x7FFF departures that would carry into the neighbouring counter.
constexpr uint32_t COUNT_WINDOW_WORDS = 2048;
constexpr uint32_t COUNT_WINDOW_LINES = 2 * COUNT_WINDOW_WORDS;
constexpr uint32_t COUNT_NONE = 0xFFFFFFFFu;

// One departure from window line `off` (block line `line`).
__device__ __forceinline__ void window_count(uint32_t* win, uint32_t off, uint32_t line,
                                             uint32_t* __restrict__ cbase, int64_t stride) {
  const uint32_t sh = (off & 1u) << 4;
  const uint32_t old = atomicAdd(win + (off >> 1), 1u << sh);
  if (__builtin_expect(((old >> sh) & 0xFFFFu) == 0x7FFFu, 0)) {
    atomicSub(win + (off >> 1), 0x8000u << sh);
    atomicAdd(cbase + count_slot(line, stride), 0x8000u);
  }
}

// The workgroup's window into the XCD's copy of the counts, one atomic per nonzero line (after
// a barrier that follows every window_count of the workgroup).
__device__ __forceinline__ void window_flush(const uint32_t* win, uint32_t base,
                                             uint32_t* __restrict__ cbase, int64_t stride) {
  for (uint32_t i = threadIdx.x; i < COUNT_WINDOW_WORDS; i += blockDim.x) {
    const uint32_t c = win[i];
    if (c & 0xFFFFu) atomicAdd(cbase + count_slot(base + 2u * i, stride), c & 0xFFFFu);
    if (c >> 16) atomicAdd(cbase + count_slot(base + 2u * i + 1u, stride), c >> 16);
  }
}

template <bool COUNT, bool SAMPLE, bool TRACE>
__device__ __forceinline__ void hop_wave(const net_view& v, uint32_t e, bool valid,
                                         uint64_t hop_budget, double t_max, const trace_view& tv,
                                         uint4* lds_wave, uint32_t lane, uint32_t* win,
                                         uint32_t win_base) {
#pragma clang fp contract(off)
  double t = INFINITY, dx = 0.0, dy = 0.0, dz = 0.0;
  uint64_t h = 0, hs = 0;
  uint32_t nd = 0, k = 0, W = 0;
  int64_t tr = 0;
  if (valid) {
    t = v.x.t_next[e];
    h = v.x.hops[e];
    dx = v.x.dx[e];
    dy = v.x.dy[e];
    dz = v.x.dz[e];
    nd = v.x.drains[e];
    hs = v.x.hash[e];
    if (SAMPLE) k = v.x.k_rec[e];
    if (TRACE && e < tv.n_trace) tr = tv.tr_n[e];
    const uint32_t R0 = (uint32_t)v.roff[v.x.site[e]];
    W = row_word(R0, v.blocks[(size_t)ROW_UNITS * R0].x);
  }
  const uint64_t h_end = h + hop_budget;
  const size_t E = v.x.n;
  // the next MSD record falls due once the clock passes t_rec = (k + 1) dt_sample
  double t_rec = INFINITY;
  if (SAMPLE && k < (uint32_t)v.n_bins) t_rec = (double)(k + 1u) * v.dt_sample;
  bool active = valid;
  bool live = false;           // when stopped: able to hop in a later launch
  uint32_t site_now = 0;       // when stopped: the site it stopped at
  bool pend = false;           // a hop waits for its target row
  uint32_t r_dw = 0;           // its dwell draw
  float px = 0.f, py = 0.f, pz = 0.f;  // position of the site it left
  double t_hop = 0.0;
  hop_words hw;
  count_cache cc;
  uint32_t* cbase = COUNT ? v.site_count + (size_t)xcd_id() * v.count_stride : nullptr;
  // the departure of the last hop is counted at the top of the next iteration, so that an
  // eviction's device atomic has a whole iteration to complete before the wave waits on its
  // next row load (one counter tracks both)
  uint32_t count_line = COUNT_NONE;
  auto count_departure = [&]() {
    const uint32_t off = count_line - win_base;
    if (off < COUNT_WINDOW_LINES) window_count(win, off, count_line, cbase, v.count_stride);
    else cc.add(count_slot(count_line, v.count_stride), cbase);
    count_line = COUNT_NONE;
  };

  coop_issue(v.blocks, W, lds_wave, lane);
  while (true) {
    // the wave issues at raised priority from its row's arrival until the next row load is out
    // (the stretch its exciton's hops wait on); the dwell and records of (B) and (C) run at the
    // normal one, so the SIMD's other waves reach their own loads first
    __builtin_amdgcn_s_setprio(2);
    const coop_row row = coop_finish(lds_wave, lane);
    if (COUNT && count_line != COUNT_NONE) count_departure();
    // (A) the hop from this site, if the exciton may still hop (scatterer::update_state,
    // scatterer.cpp:17-30), and the load of the row it leads to
    const bool can = active && h < h_end && !trapped(row.n, row.gamma);
    uint32_t tg = 0, r_next = 0, W_next = W;
    if (can) {
      uint32_t w_sel, w_dw;
      hw.get(v.seed, e, h, w_sel, w_dw);
      const double dice = div_rand_max(row.gamma * (double)r31(w_sel));
      const uint32_t idx = select_entry(v.blocks, W, row.c, row.n, dice);
      tg = idx < ROW_INLINE ? target_lds(lds_wave, lane, idx) : target_wide(v.blocks, W, row.n, idx);
      r_next = nonzero_draw1(w_dw, v.seed, e, h, STREAM_HOP_REDRAW);
      W_next = (tg & EDGE_DRAIN_BIT) ? v.src_roff[r31(draw4(v.seed, e, h, STREAM_REINJECT).v[0]) % v.n_src]
                                     : (tg & ~EDGE_DRAIN_BIT);
    }
    // a lane whose exciton has stopped never reads its row again: it loads block line 0, which
    // every such lane of the wave shares, instead of its own row
    coop_issue(v.blocks, active ? W_next : 0u, lds_wave, lane);
    __builtin_amdgcn_s_setprio(0);
    // (B) the hop into this site finishes: dwell at the new site (particle.cpp:183 -> ff_time)
    if (pend) {
      dx = dx + min_image((double)row.x - (double)px, v.half_per[0]);
      dy = dy + min_image((double)row.y - (double)py, v.half_per[1]);
      dz = dz + min_image((double)row.z - (double)pz, v.half_per[2]);
      hs = (hs ^ (uint64_t)row.site) * FNV_PRIME;
      t = t + dwell_time(row.n, row.gamma, r_dw);
      if (TRACE && e < tv.n_trace && tr < tv.tr_max) {
        tv.tr_site[(size_t)e * tv.tr_max + tr] = (int32_t)row.site;
        tv.tr_time[(size_t)e * tv.tr_max + tr] = t_hop;
        ++tr;
      }
      pend = false;
    }
    if (SAMPLE && active) {
      while (t_rec < t) {
        const size_t r = (size_t)(k - (uint32_t)v.bin0) * E + e;
        v.rec_dx[r] = dx;
        v.rec_dy[r] = dy;
        v.rec_dz[r] = dz;
        v.rec_drain[r] = nd;
        ++k;
        t_rec = k < (uint32_t)v.n_bins ? (double)(k + 1u) * v.dt_sample : INFINITY;
      }
    }
    // (C) the hop of (A) happens at t if t <= t_max; otherwise the exciton stops here
    const bool hop = can && t <= t_max;
    if (active && !hop) {
      active = false;
      site_now = row.site;
      live = !trapped(row.n, row.gamma) && t <= t_max;
    }
    if (hop) {
      if (COUNT) count_line = W & TGT_LINE_MASK;
      t_hop = t;
      if (tg & EDGE_DRAIN_BIT) {
        // drain: the dwell drawn at the drain site, then re-injection keeping displacement and
        // dwell (kubo_step, src/monte_carlo/monte_carlo.cpp:330-336)
        const uint4* bd = v.blocks + (size_t)ROW_UNITS * (tg & TGT_LINE_MASK);
        const uint4 hd = bd[0], pd = bd[7];
        dx = dx + min_image((double)__uint_as_float(pd.x) - (double)row.x, v.half_per[0]);
        dy = dy + min_image((double)__uint_as_float(pd.y) - (double)row.y, v.half_per[1]);
        dz = dz + min_image((double)__uint_as_float(pd.z) - (double)row.z, v.half_per[2]);
        hs = (hs ^ (uint64_t)hd.y) * FNV_PRIME;
        t = t + dwell_time(hd.x, __hiloint2double((int)hd.w, (int)hd.z), r_next);
        ++nd;
        const uint32_t src_site = v.blocks[(size_t)ROW_UNITS * (W_next & TGT_LINE_MASK)].y;
        hs = (hs ^ ((uint64_t)src_site | (1ull << 32))) * FNV_PRIME;
        if (TRACE && e < tv.n_trace && tr < tv.tr_max) {
          tv.tr_site[(size_t)e * tv.tr_max + tr] = (int32_t)src_site;
          tv.tr_time[(size_t)e * tv.tr_max + tr] = t_hop;
          ++tr;
        }
      } else {
        pend = true;
        r_dw = r_next;
        px = row.x;
        py = row.y;
        pz = row.z;
      }
      W = W_next;
      ++h;
    }
    if (__ballot(active) == 0) break;
  }
  // the last issued load lands in this wave's LDS rows: wait for it before the wave moves on
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (COUNT && count_line != COUNT_NONE) count_departure();
  if (COUNT) cc.flush(cbase);
  if (v.live) {
    // excitons that a further launch could move (the budget aside)
    const uint64_t b = __ballot(valid && live), due = __ballot(valid && t <= t_max);
    if (lane == 0u) add_live(v.live, b, due);
  }
  if (!valid) return;
  v.x.site[e] = (int32_t)site_now;
  v.x.t_next[e] = t;
  v.x.hops[e] = h;
  v.x.dx[e] = dx;
  v.x.dy[e] = dy;
  v.x.dz[e] = dz;
  v.x.drains[e] = nd;
  v.x.hash[e] = hs;
  if (SAMPLE) v.x.k_rec[e] = k;
  if (TRACE && e < tv.n_trace) tv.tr_n[e] = tr;
}

// The hops of one wave's excitons (event-driven form of particle::step,
// src/monte_carlo/particle.cpp:57-80) with drift along the tubes for v > 0, built like hop_wave.
// Below ~100,000 excitons the chain of one iteration bounds the kernel (~330 vector and ~210 scalar
// instructions), above it their issue; so the next row's load goes out before the dwell, the records
// and the flight are computed: on a guess whether the flight ends on its leg (the dwell in single
// precision), or exactly when the flight's time is known already.  The guess decides only which row
// is loaded; where it is wrong the lane spends an iteration on loading the right one.  An iteration
// takes a lane one site on, by a hop or along the tube, so lanes in a long flight hold back no others.
// `c` is the view's copy in LDS, for what few iterations need: as kernel arguments those pointers
// would hold scalar registers throughout (~100 were spilled to lanes of vector registers).
// 1,000 hops on 50,051 sites at 2e5 m/s, with counts and records / without, in ms: 100,003 excitons
// 3.27 / 2.49, 1 M 22.7 / 13.3; a lane with its own gathers through flight and hop 3.65 / 2.96 and
// 27.5 / 18.9.  Three waves per SIMD instead of two spill 45 registers with counts and records:
// 4.93 and 32.9.
template <bool COUNT, bool SAMPLE, bool TRACE>
__device__ __forceinline__ void hop_wave_fly(const net_view& v, uint32_t e, bool valid,
                                             uint64_t hop_budget, double t_max,
                                             const trace_view& tv, uint4* lds_wave, uint32_t lane,
                                             uint32_t* win, uint32_t win_base, const net_view& c) {
#pragma clang fp contract(off)
  double t = INFINITY, tl = 0.0, so = 0.0, dx = 0.0, dy = 0.0, dz = 0.0;
  uint64_t h = 0, hs = 0;
  uint32_t hd = 0, nd = 0, k = 0, W = 0;
  int64_t tr = 0;
  if (valid) {
    t = c.x.t_next[e];
    tl = c.x.t_last[e];
    so = c.x.s_off[e];
    hd = (uint32_t)c.x.heading[e];
    h = c.x.hops[e];
    dx = c.x.dx[e];
    dy = c.x.dy[e];
    dz = c.x.dz[e];
    nd = c.x.drains[e];
    hs = c.x.hash[e];
    if (SAMPLE) k = c.x.k_rec[e];
    if (TRACE && e < tv.n_trace) tr = tv.tr_n[e];
    const uint32_t R0 = (uint32_t)c.roff[c.x.site[e]];
    W = row_word(R0, v.blocks[(size_t)ROW_UNITS * R0].x);
  }
  const uint64_t h_end = h + hop_budget;
  double t_rec = INFINITY;
  if (SAMPLE && k < (uint32_t)v.n_bins) t_rec = (double)(k + 1u) * v.dt_sample;
  bool active = valid;
  uint32_t site_now = 0;       // when stopped: the site it stopped at
  bool pend = false;           // a hop into this site is to be finished
  uint32_t r_dw = 0;           // its dwell draw
  float px = 0.f, py = 0.f, pz = 0.f;  // position of the site it left
  bool flown = false;          // on a flight whose remaining time is tau
  bool reload = false;         // the row on its way is not the lane's: W is to be loaded
  double tau = 0.0;
  uint32_t passes = 0, fly_drains = 0;  // sites and drains passed on the flight
  // the state before the flight, restored when it exceeds the pass bound
  double so0 = 0.0, dx0 = 0.0, dy0 = 0.0, dz0 = 0.0;
  uint64_t hs0 = 0;
  uint32_t hd0 = 0, nd0 = 0, site0 = 0;
  hop_words hw;
  count_cache cc;
  uint32_t* cbase = COUNT ? v.site_count + (size_t)xcd_id() * v.count_stride : nullptr;
  uint32_t count_line = COUNT_NONE;  // counted at the top of the next iteration, as in hop_wave
  auto count_departure = [&]() {
    const uint32_t off = count_line - win_base;
    if (off < COUNT_WINDOW_LINES) window_count(win, off, count_line, cbase, v.count_stride);
    else cc.add(count_slot(count_line, v.count_stride), cbase);
    count_line = COUNT_NONE;
  };

  coop_issue(v.blocks, W, lds_wave, lane);
  // the next leg as loaded: unpacked only after the row has arrived, or the wave would wait for it
  // where it is issued
  const uint4* at = leg_of(v, W, hd);
  uint4 leg_p = at[0], leg_q = at[1];
  while (true) {
    const coop_row row = coop_finish(lds_wave, lane);
    const fly_leg leg = leg_from_units(leg_p, leg_q);
    if (COUNT && count_line != COUNT_NONE) count_departure();
    // (A) where the lane goes next, guessed, and the load of that row: the hop from this site if
    // the flight through the dwell is taken to end on its leg, else the leg's site
    const bool on = active && !reload;
    const bool linked = leg.word != LINK_NONE;  // particle.cpp:11-12
    double need = 0.0;
    bool stay = true;
    if (on && linked) {
      need = (leg.len - so) / v.velocity;
      if (flown) {
        stay = !(need < tau);
      } else {
        // the dwell in single precision: a wrong guess costs an iteration, nothing else
        const float guess = pend ? -__log2f((float)r_dw * 0x1p-31f) * 0.6931472f / (float)row.gamma
                                 : (float)(t - tl);
        stay = !((float)need < guess);
      }
    }
    uint32_t tg = 0, r_next = 0, W_next = W;
    const bool can = on && stay && h < h_end && !trapped(row.n, row.gamma);
    if (can) {
      // event selection (scatterer::update_state, scatterer.cpp:17-30)
      uint32_t w_sel, w_dw;
      hw.get(v.seed, e, h, w_sel, w_dw);
      const double dice = div_rand_max(row.gamma * (double)r31(w_sel));
      const uint32_t idx = select_entry(v.blocks, W, row.c, row.n, dice);
      tg = idx < ROW_INLINE ? target_lds(lds_wave, lane, idx) : target_wide(v.blocks, W, row.n, idx);
      r_next = nonzero_draw1(w_dw, v.seed, e, h, STREAM_HOP_REDRAW);
      W_next = tg & ~EDGE_DRAIN_BIT;
      if (tg & EDGE_DRAIN_BIT) {
        W_next = c.src_roff[r31(draw4(v.seed, e, h, STREAM_REINJECT).v[0]) % c.n_src];
      }
    } else if (on && !stay) {
      W_next = leg.word & ~EDGE_DRAIN_BIT;
      if (leg.word & EDGE_DRAIN_BIT) {
        W_next = c.src_roff[r31(draw4(v.seed, e, h, STREAM_FLY_DRAIN + fly_drains).v[0]) % c.n_src];
      }
    }
    const uint32_t hd_next = on && linked ? leg.heading : hd;
    // a lane whose exciton has stopped loads block line 0, which every such lane shares
    coop_issue(v.blocks, active ? W_next : 0u, lds_wave, lane);
    at = leg_of(v, active ? W_next : 0u, hd_next);
    leg_p = at[0];
    leg_q = at[1];
    reload = false;
    // (B) the hop into this site finishes: dwell at the new site (particle.cpp:183 -> ff_time)
    if (pend && on) {
      dx = dx + min_image((double)row.x - (double)px, v.half_per[0]);
      dy = dy + min_image((double)row.y - (double)py, v.half_per[1]);
      dz = dz + min_image((double)row.z - (double)pz, v.half_per[2]);
      hs = (hs ^ (uint64_t)row.site) * FNV_PRIME;
      if (TRACE && e < tv.n_trace && tr < tv.tr_max) {
        tv.tr_site[(size_t)e * tv.tr_max + tr] = (int32_t)row.site;
        tv.tr_time[(size_t)e * tv.tr_max + tr] = t;
        ++tr;
      }
      t = t + dwell_time(row.n, row.gamma, r_dw);
      pend = false;
    }
    if (on && !flown) {
      if (SAMPLE) {
        while (t_rec < t) {  // the flight from the last event up to t_rec
          const double tau_r = t_rec - tl;
          double gx = dx, gy = dy, gz = dz;
          uint32_t gd = nd;
          if (!linked || !(need < tau_r)) {
            const double s_r = linked ? so + v.velocity * tau_r : so;
            if (s_r != 0.0) {
              const double q = s_r / leg.len;
              gx = dx + min_image((double)leg.x - (double)row.x, v.half_per[0]) * q;
              gy = dy + min_image((double)leg.y - (double)row.y, v.half_per[1]) * q;
              gz = dz + min_image((double)leg.z - (double)row.z, v.half_per[2]) * q;
            }
          } else {
            flight_state g{W, row.site, row.x, row.y, row.z, so, hd, dx, dy, dz, nd, hs};
            fly_leg gl = leg;
            net_view fv = v;
            fv.src_roff = c.src_roff;
            fv.n_src = c.n_src;
            if (!fly(fv, g, gl, tau_r, e, h)) {
              atomicOr(c.fly_err, 1);
              break;
            }
            double ox, oy, oz;
            fly_offset(c, g, gl, ox, oy, oz);
            gx = g.dx + ox;
            gy = g.dy + oy;
            gz = g.dz + oz;
            gd = g.nd;
          }
          const size_t r = (size_t)(k - (uint32_t)c.bin0) * c.x.n + e;
          c.rec_dx[r] = gx;
          c.rec_dy[r] = gy;
          c.rec_dz[r] = gz;
          c.rec_drain[r] = gd;
          ++k;
          t_rec = k < (uint32_t)c.n_bins ? (double)(k + 1u) * c.dt_sample : INFINITY;
        }
      }
      if (h >= h_end || !(t <= t_max) || !(t < INFINITY)) {
        active = false;
        site_now = row.site;
      } else {
        // fly through the dwell, then hop from the site reached (particle.cpp:62-75)
        tau = t - tl;
        so0 = so;
        dx0 = dx;
        dy0 = dy;
        dz0 = dz;
        hs0 = hs;
        hd0 = hd;
        nd0 = nd;
        site0 = row.site;
      }
    }
    // (C) what (A) guessed, if it holds; otherwise the row again, with the flight's time known
    if (on && active) {
      if (linked && passes == FLY_MAX_PASSES) {
        atomicOr(c.fly_err, 1);
        so = so0;
        dx = dx0;
        dy = dy0;
        dz = dz0;
        hs = hs0;
        hd = hd0;
        nd = nd0;
        site_now = site0;
        active = false;
      } else if (linked && stay == (need < tau)) {
        flown = reload = true;
      } else if (!stay) {  // passes the leg's site
        tau = tau - need;
        dx = dx + min_image((double)leg.x - (double)row.x, v.half_per[0]);
        dy = dy + min_image((double)leg.y - (double)row.y, v.half_per[1]);
        dz = dz + min_image((double)leg.z - (double)row.z, v.half_per[2]);
        so = 0.0;
        hs = (hs ^ ((uint64_t)leg.site | (2ull << 32))) * FNV_PRIME;
        if (leg.word & EDGE_DRAIN_BIT) {
          ++nd;
          ++fly_drains;
          const uint32_t src_site = v.blocks[(size_t)ROW_UNITS * (W_next & TGT_LINE_MASK)].y;
          hs = (hs ^ ((uint64_t)src_site | (1ull << 32))) * FNV_PRIME;
        }
        ++passes;
        flown = true;
        hd = hd_next;
        W = W_next;
      } else {  // ends on this segment (particle.cpp:46-49)
        if (linked) so = so + v.velocity * tau;
        hd = hd_next;
        flown = false;
        passes = fly_drains = 0u;
        if (!can) {
          // no rates here: the event leaves the exciton in place (scatterer.cpp:14-15) and no dwell
          // ends again; it counts as a hop so that later flights draw on fresh counters
          tl = t;
          t = INFINITY;
          ++h;
          hw.have = false;
        } else {
          if (COUNT) count_line = W & TGT_LINE_MASK;
          so = 0.0;
          tl = t;
          if (tg & EDGE_DRAIN_BIT) {
            // drain: the dwell drawn at the drain site, then re-injection keeping displacement and
            // dwell (kubo_step, src/monte_carlo/monte_carlo.cpp:330-336)
            const uint4* bd = v.blocks + (size_t)ROW_UNITS * (tg & TGT_LINE_MASK);
            const uint4 hdr = bd[0], pd = bd[7];
            dx = dx + min_image((double)__uint_as_float(pd.x) - (double)row.x, v.half_per[0]);
            dy = dy + min_image((double)__uint_as_float(pd.y) - (double)row.y, v.half_per[1]);
            dz = dz + min_image((double)__uint_as_float(pd.z) - (double)row.z, v.half_per[2]);
            hs = (hs ^ (uint64_t)hdr.y) * FNV_PRIME;
            ++nd;
            const uint32_t src_site = v.blocks[(size_t)ROW_UNITS * (W_next & TGT_LINE_MASK)].y;
            hs = (hs ^ ((uint64_t)src_site | (1ull << 32))) * FNV_PRIME;
            if (TRACE && e < tv.n_trace && tr < tv.tr_max) {
              tv.tr_site[(size_t)e * tv.tr_max + tr] = (int32_t)src_site;
              tv.tr_time[(size_t)e * tv.tr_max + tr] = t;
              ++tr;
            }
            t = t + dwell_time(hdr.x, __hiloint2double((int)hdr.w, (int)hdr.z), r_next);
          } else {
            pend = true;
            r_dw = r_next;
            px = row.x;
            py = row.y;
            pz = row.z;
          }
          ++h;
          W = W_next;
        }
      }
    }
    if (__ballot(active) == 0) break;
  }
  // the last issued load lands in this wave's LDS rows: wait for it before the wave moves on
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (COUNT && count_line != COUNT_NONE) count_departure();
  if (COUNT) cc.flush(cbase);
  if (uint32_t* live = c.live) {
    const uint64_t b = __ballot(valid && t <= t_max && t < INFINITY);
    if (lane == 0u && b != 0ull) atomicAdd(live, (uint32_t)__popcll(b));
  }
  if (!valid) return;
  c.x.site[e] = (int32_t)site_now;
  c.x.t_next[e] = t;
  c.x.hops[e] = h;
  c.x.dx[e] = dx;
  c.x.dy[e] = dy;
  c.x.dz[e] = dz;
  c.x.drains[e] = nd;
  c.x.hash[e] = hs;
  if (SAMPLE) c.x.k_rec[e] = k;
  if (TRACE && e < tv.n_trace) tv.tr_n[e] = tr;
  c.x.s_off[e] = so;
  c.x.t_last[e] = tl;
  c.x.heading[e] = (uint8_t)hd;
}

// Position of this thread in the sorted exciton order.  Workgroups are dealt to the XCDs in turn,
// so workgroup b takes the b%8-th eighth of the order: each XCD's L2 serves excitons that sit on
// neighbouring blocks.  gridDim.x is a multiple of KMC_COUNT_COPIES.
__device__ __forceinline__ uint32_t xcd_position() {
  const uint32_t per_xcd = gridDim.x / KMC_COUNT_COPIES;
  const uint32_t chunk = (blockIdx.x % KMC_COUNT_COPIES) * per_xcd + blockIdx.x / KMC_COUNT_COPIES;
  return chunk * blockDim.x + threadIdx.x;
}

// One network: thread -> position -> exciton perm[position] (its id keys every draw, so the order
// changes nothing but locality).
template <bool COUNT, bool SAMPLE, bool TRACE>
__global__ __launch_bounds__(256, 4) void k_hop(hop_args a) {
  __shared__ uint4 rows[4 * 64 * ROW_UNITS];  // 8 KB of staged rows per wave
  __shared__ uint32_t win[COUNT_WINDOW_WORDS]; // 8 KB: the workgroup's departure-count window
  // the positions taken: all excitons, or the ones not idle in a clock-bounded launch (sorted
  // first), dealt in eighths to the XCDs like all of them
  uint32_t pos, n;
  if (a.n_alive) {
    n = *a.n_alive;
    const uint32_t per_xcd = ((n + 255u) / 256u + KMC_COUNT_COPIES - 1) / KMC_COUNT_COPIES;
    const uint32_t rank = blockIdx.x / KMC_COUNT_COPIES;
    pos = rank < per_xcd
              ? ((blockIdx.x % KMC_COUNT_COPIES) * per_xcd + rank) * blockDim.x + threadIdx.x
              : 0xFFFFFFFFu;
  } else {
    n = (uint32_t)a.v.x.n;
    pos = xcd_position();
  }
  const uint32_t lane = threadIdx.x & 63u;
  const bool wave_live = __builtin_amdgcn_readfirstlane(pos - lane) < n;
  const bool valid = pos < n;
  const uint32_t e = valid ? (a.perm ? a.perm[pos] : pos) : 0u;
  uint4* lds_wave = rows + 64u * ROW_UNITS * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if constexpr (!COUNT) {
    if (wave_live)
      hop_wave<COUNT, SAMPLE, TRACE>(a.v, e, valid, a.hop_budget, a.t_max, a.tv, lds_wave, lane,
                                     nullptr, 0u);
  } else {
    // The workgroup's excitons are consecutive in the order sorted by block line, and their
    // hops in one sub-launch stay mostly among nearby blocks: departures from the window's
    // lines around the first one's line are summed in LDS and flushed once, per line, at the end.
    for (uint32_t i = threadIdx.x; i < COUNT_WINDOW_WORDS; i += blockDim.x) win[i] = 0u;
    const uint32_t p0 = pos - threadIdx.x;
    uint32_t base = 0u;
    if (p0 < n) {
      const uint32_t e0 = a.perm ? a.perm[p0] : p0;
      const uint32_t L0 = (uint32_t)a.v.roff[a.v.x.site[e0]];
      base = L0 > COUNT_WINDOW_LINES / 2 ? L0 - COUNT_WINDOW_LINES / 2 : 0u;
    }
    __syncthreads();
    if (wave_live)
      hop_wave<COUNT, SAMPLE, TRACE>(a.v, e, valid, a.hop_budget, a.t_max, a.tv, lds_wave, lane,
                                     win, base);
    __syncthreads();
    window_flush(win, base, a.v.site_count + (size_t)xcd_id() * a.v.count_stride,
                 a.v.count_stride);
  }
}

// ---------------------------------------------------------------------------------------------
// Few excitons (k_hop_rows).  With less than a wave per SIMD, k_hop's iteration takes its own
// latency: LDS round trips, lane exchanges, ten Philox rounds and a logarithm one after another
// in a single wave, ~3,500 cycles per hop, of which the row load itself is hidden; the chip is
// idle.  What bounds this form is the same chain, shortened: ~1,100 cycles per hop, a quarter of
// them the row's L2 latency (76,543 sites, 1,250 hops with counts: 1,000 excitons 1.86 -> 0.57 ms,
// 16,384 excitons 1.92 -> 0.84 ms).  Each exciton has a row of 16 lanes, four excitons to a wave.
// The lanes hold the exciton's 128-byte block line between them (8 bytes each), so a selection is a
// comparison per lane and a count of the ballot's bits, with DPP row broadcasts instead of LDS
// staging.  Only the chain that leads
// from row to row runs hop by hop; a batch of ROW_BATCH = 16 hops then has its draws, dwells and
// displacements computed side by side, lane j for hop j, and folded into the exciton's sums in
// hop order (the operations and their order are those of hop_wave, so are the bits).  Hops
// selected past t_max are dropped when the batch is folded; a batch costs its hops, so a launch of
// a hop or two ends it early, and the first batch of a run up to a time, which may end within a few
// hops, has four (64 excitons, one hop: 31.6 -> 29.3 us a call, 27.5 with k_hop).
constexpr uint32_t ROW_BATCH = 16, ROW_FIRST = 4;

struct __align__(16) batch_lds {
  uint4 reached[4][ROW_BATCH][2];  // per exciton and hop: {n, site, Gamma}, {x, y, z, -} of the row
  double inc[4][ROW_BATCH][4];     // dwell, displacement x, y, z of the hop
};

// Value of lane L of the lane's row of 16 (v_mov_b32 with row_newbcast).
template <int L>
__device__ __forceinline__ uint32_t row_bcast(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x150 + L, 0xF, 0xF, true);
}
template <int L>
__device__ __forceinline__ double row_bcast(double x) {
  return __hiloint2double((int)row_bcast<L>((uint32_t)__double2hiint(x)),
                          (int)row_bcast<L>((uint32_t)__double2loint(x)));
}

// LDS written by some lanes of the wave and read by others: in order within the wave, which
// the compiler must keep.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The chain of one batch.
struct row_chain {
  uint2 raw;        // the lane's 8 bytes of the current row's first line
  uint2 more;       // and of its second line, for a row word with TGT_WIDE_BIT
  uint32_t W;       // its row word
  uint32_t cnt;     // hops selected in this batch
  bool run;
  uint32_t my_tg, my_W;  // lane j: target word and departure row word of hop j
};

// The lines of row word c.W, 8 bytes per lane.
__device__ __forceinline__ void load_lines(const net_view& v, row_chain& c, uint32_t l) {
  const uint32_t off = (c.W & TGT_LINE_MASK) * (uint32_t)(16u * ROW_UNITS) + 8u * l;
  const char* b = reinterpret_cast<const char*>(v.blocks);
  c.raw = *reinterpret_cast<const uint2*>(b + off);
  if (c.W & TGT_WIDE_BIT) c.more = *reinterpret_cast<const uint2*>(b + off + 16u * ROW_UNITS);
}

// Hop J of the batch; false when no exciton of the wave makes it.
template <int J>
__device__ __forceinline__ bool row_step(const net_view& v, row_chain& c, uint32_t e, uint64_t h0,
                                         uint32_t left, double r_sel, uint32_t l, uint32_t g,
                                         batch_lds* s) {
#pragma clang fp contract(off)
  if (J > 0) {
    // the row that hop J - 1 reached: header and position (lanes 0, 1, 14, 15)
    if (l < 2u || l >= 14u) reinterpret_cast<uint2*>(&s->reached[g][J > 0 ? J - 1 : 0][0])[l & 3u] = c.raw;
  }
  const uint32_t n = row_bcast<0>(c.raw.x);
  const double mine = __hiloint2double((int)c.raw.y, (int)c.raw.x);
  const double gamma = row_bcast<1>(mine);
  const bool can = c.run && (uint32_t)J < left && !trapped(n, gamma);
  // a short batch ends here; asked at two hops only, the other steps stay one block of instructions
  if constexpr (J == 1 || J == (int)ROW_FIRST) {
    if (__ballot(can) == 0ull) return false;
  }
  // the lanes 2..9 hold the inline cumulative rates: their count <= dice is the selected entry
  const double dice = div_rand_max(gamma * row_bcast<J>(r_sel));
  const uint64_t le = __ballot(mine <= dice);
  uint32_t idx = (uint32_t)__popc((uint32_t)(le >> (16u * g)) & 0x3FCu);
  // targets 0..7 sit two to a lane in the lanes 10..13
  const int src = (int)(4u * (16u * g + 10u + ((idx & 7u) >> 1)));
  const uint32_t t0 = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)c.raw.x);
  const uint32_t t1 = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)c.raw.y);
  uint32_t tg = (idx & 1u) ? t1 : t0;
  const bool wide = can && idx >= ROW_INLINE;
  if (__ballot(wide) != 0ull) {
    // the continuation line came with the first one: cum[8..n), then tgt[8..n), of a row with up
    // to 18 entries
    const uint32_t m = n - ROW_INLINE;
    const bool one = m <= 10u;
    const uint64_t lw = __ballot(wide && one && l + 1u < m &&
                                 __hiloint2double((int)c.more.y, (int)c.more.x) <= dice);
    const uint32_t word = 2u * m + (uint32_t)__popc((uint32_t)(lw >> (16u * g)) & 0xFFFFu);
    const int at = (int)(4u * (16u * g + ((word >> 1) & 15u)));
    const uint32_t w0 = (uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)c.more.x);
    const uint32_t w1 = (uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)c.more.y);
    if (wide) tg = (word & 1u) ? w1 : w0;
    // longer rows sixteen entries at a time
    const char* ce = reinterpret_cast<const char*>(v.blocks) +
                     ((size_t)(c.W & TGT_LINE_MASK) + 1u) * (16u * ROW_UNITS);
    bool left_over = wide && !one;
    for (uint32_t q = 0; __ballot(left_over) != 0ull; q += 16u) {
      const uint32_t k = q + l;
      double ck = INFINITY;
      uint32_t tk = 0u;
      if (left_over && k < m) {
        if (k + 1u < m) ck = *reinterpret_cast<const double*>(ce + 8u * (size_t)k);
        tk = *reinterpret_cast<const uint32_t*>(ce + 8u * (size_t)m + 4u * (size_t)k);
      }
      const uint64_t lk = __ballot(ck <= dice);
      const uint32_t add = (uint32_t)__popc((uint32_t)(lk >> (16u * g)) & 0xFFFFu);
      const uint32_t tw =
          (uint32_t)__builtin_amdgcn_ds_bpermute((int)(4u * (16u * g + (add & 15u))), (int)tk);
      if (left_over && add < 16u) {
        tg = tw;
        left_over = false;
      }
    }
  }
  uint32_t Wn = tg & ~EDGE_DRAIN_BIT;
  if (can && (tg & EDGE_DRAIN_BIT))
    Wn = v.src_roff[r31(draw4(v.seed, e, h0 + (uint32_t)J, STREAM_REINJECT).v[0]) % v.n_src];
  if (l == (uint32_t)J) {
    c.my_tg = tg;
    c.my_W = c.W;
  }
  c.run = can;
  if (can) {
    c.W = Wn;
    ++c.cnt;
    load_lines(v, c, l);
  }
  return true;
}

template <int... J>
__device__ __forceinline__ void row_steps(std::integer_sequence<int, J...>, const net_view& v,
                                          row_chain& c, uint32_t e, uint64_t h0, uint32_t left,
                                          double r_sel, uint32_t l, uint32_t g, batch_lds* s) {
  (void)(row_step<J>(v, c, e, h0, left, r_sel, l, g, s) && ...);
}

// Visit hash over the sites the batch's hops reached, in hop order (none of them a drain).
template <int... J>
__device__ __forceinline__ uint64_t row_hash(std::integer_sequence<int, J...>, uint64_t hs,
                                             uint32_t site, uint32_t cnt) {
  ((hs = (uint32_t)J < cnt ? (hs ^ (uint64_t)row_bcast<J>(site)) * FNV_PRIME : hs), ...);
  return hs;
}

template <bool COUNT, bool SAMPLE, bool TRACE>
__device__ __forceinline__ void hop_rows(const net_view& v, uint32_t e, bool valid,
                                         uint64_t hop_budget, double t_max, const trace_view& tv,
                                         batch_lds* s, uint32_t lane, uint32_t* win,
                                         uint32_t win_base, uint32_t win_lines) {
#pragma clang fp contract(off)
  using hops16 = std::make_integer_sequence<int, (int)ROW_BATCH>;
  const uint32_t l = lane & 15u, g = lane >> 4;
  // the exciton's state, the same in its 16 lanes
  double t = INFINITY, dx = 0.0, dy = 0.0, dz = 0.0;
  uint64_t h = 0, hs = 0;
  uint32_t nd = 0, k = 0;
  int64_t tr = 0;
  row_chain c{};
  if (valid) {
    t = v.x.t_next[e];
    h = v.x.hops[e];
    dx = v.x.dx[e];
    dy = v.x.dy[e];
    dz = v.x.dz[e];
    nd = v.x.drains[e];
    hs = v.x.hash[e];
    if (SAMPLE) k = v.x.k_rec[e];
    if (TRACE && e < tv.n_trace) tr = tv.tr_n[e];
    const uint32_t R0 = (uint32_t)v.roff[v.x.site[e]];
    c.W = row_word(R0, v.blocks[(size_t)ROW_UNITS * R0].x);
  }
  load_lines(v, c, l);
  uint32_t n = row_bcast<0>(c.raw.x), site = row_bcast<0>(c.raw.y);
  double gamma = row_bcast<1>(__hiloint2double((int)c.raw.y, (int)c.raw.x));
  float px = __uint_as_float(row_bcast<14>(c.raw.x)), py = __uint_as_float(row_bcast<14>(c.raw.y)),
        pz = __uint_as_float(row_bcast<15>(c.raw.x));
  const uint64_t h_end = h + hop_budget;
  const size_t E = v.x.n;
  double t_rec = INFINITY;
  if (SAMPLE && k < (uint32_t)v.n_bins) t_rec = (double)(k + 1u) * v.dt_sample;
  uint32_t* cbase = COUNT ? v.site_count + (size_t)xcd_id() * v.count_stride : nullptr;
  // the MSD records that fall due before the pending hop at t
  auto records = [&]() {
    while (t_rec < t) {
      const size_t r = (size_t)(k - (uint32_t)v.bin0) * E + e;
      if (l == 0u) {
        v.rec_dx[r] = dx;
        v.rec_dy[r] = dy;
        v.rec_dz[r] = dz;
        v.rec_drain[r] = nd;
      }
      ++k;
      t_rec = k < (uint32_t)v.n_bins ? (double)(k + 1u) * v.dt_sample : INFINITY;
    }
  };
  if (SAMPLE && valid) records();
  bool active = valid && h < h_end && t <= t_max && !trapped(n, gamma);
  // the chain finds out only after its batch that t_max was passed
  uint32_t batch = t_max < INFINITY ? ROW_FIRST : ROW_BATCH;

  while (__ballot(active) != 0ull) {
    // lane j's draws for hop h + j (one Philox call holds the words of two hops)
    const uint64_t hj = h + l;
    const u32x4 w = draw4(v.seed, e, hj >> 1, STREAM_HOP);
    const bool odd = (hj & 1u) != 0u;
    const double r_sel = (double)r31(odd ? w.v[2] : w.v[0]);
    const uint32_t r_dw = nonzero_draw1(odd ? w.v[3] : w.v[1], v.seed, e, hj, STREAM_HOP_REDRAW);
    const uint64_t left = active ? h_end - h : 0u;
    const uint32_t most = left < batch ? (uint32_t)left : batch;
    batch = ROW_BATCH;
    c.cnt = 0u;
    c.run = active;
    row_steps(hops16{}, v, c, e, h, most, r_sel, l, g, s);
    if (l < 2u || l >= 14u) reinterpret_cast<uint2*>(&s->reached[g][ROW_BATCH - 1][0])[l & 3u] = c.raw;
    wave_lds_fence();
    // lane j: hop j's dwell at the site reached and its displacement
    const bool made = l < c.cnt;
    const uint4 q0 = s->reached[g][l][0], q1 = s->reached[g][l][1];
    const uint4 p1 = s->reached[g][l > 0u ? l - 1u : 0u][1];
    const float fx = l > 0u ? __uint_as_float(p1.x) : px, fy = l > 0u ? __uint_as_float(p1.y) : py,
                fz = l > 0u ? __uint_as_float(p1.z) : pz;
    const bool drained = made && (c.my_tg & EDGE_DRAIN_BIT);
    uint4 hd = q0, pd = q1;  // the hop's target: the row reached, or the drain site it re-injected from
    if (drained) {
      const uint4* bd = v.blocks + (size_t)ROW_UNITS * (c.my_tg & TGT_LINE_MASK);
      hd = bd[0];
      pd = bd[7];
    }
    double i_t = 0.0, i_x = 0.0, i_y = 0.0, i_z = 0.0;
    if (made) {
      i_t = dwell_time(hd.x, __hiloint2double((int)hd.w, (int)hd.z), r_dw);
      i_x = min_image((double)__uint_as_float(pd.x) - (double)fx, v.half_per[0]);
      i_y = min_image((double)__uint_as_float(pd.y) - (double)fy, v.half_per[1]);
      i_z = min_image((double)__uint_as_float(pd.z) - (double)fz, v.half_per[2]);
    }
    s->inc[g][l][0] = i_t;
    s->inc[g][l][1] = i_x;
    s->inc[g][l][2] = i_y;
    s->inc[g][l][3] = i_z;
    wave_lds_fence();
    // the sums in hop order: lane q of each four takes quantity q (an addition of zero for the
    // hops not made changes nothing)
    const uint32_t q = l & 3u;
    double acc = q == 0u ? t : q == 1u ? dx : q == 2u ? dy : dz;
#pragma unroll
    for (uint32_t j = 0; j < ROW_BATCH; ++j) acc = acc + s->inc[g][j][q];
    const double t_end = row_bcast<0>(acc);
    const uint64_t drain_mask = __ballot(drained);
    // no record falls due and no hop passes t_max before the batch's end, and nobody drained
    const bool plain = !TRACE && !(t_rec < t_end) && t_end <= t_max;
    uint32_t done = c.cnt;
    if (__ballot(active && !plain) == 0ull && drain_mask == 0ull) {
      t = t_end;
      dx = row_bcast<1>(acc);
      dy = row_bcast<2>(acc);
      dz = row_bcast<3>(acc);
      hs = row_hash(hops16{}, hs, q0.y, c.cnt);
    } else {
      done = 0u;
      while (true) {
        const bool go = done < c.cnt && t <= t_max;
        if (__ballot(go) == 0ull) break;
        if (go) {
          const double* inc = s->inc[g][done];
          const uint32_t at = 16u * g + done;
          const uint32_t tg = (uint32_t)__shfl((int)c.my_tg, (int)at, 64);
          const uint32_t to = (uint32_t)__shfl((int)hd.y, (int)at, 64);
          const uint32_t reached = s->reached[g][done][0].y;
          const double t_hop = t;
          dx = dx + inc[1];
          dy = dy + inc[2];
          dz = dz + inc[3];
          hs = (hs ^ (uint64_t)to) * FNV_PRIME;
          t = t + inc[0];
          if (tg & EDGE_DRAIN_BIT) {
            ++nd;
            hs = (hs ^ ((uint64_t)reached | (1ull << 32))) * FNV_PRIME;
          }
          if (TRACE && e < tv.n_trace && tr < tv.tr_max) {
            if (l == 0u) {
              tv.tr_site[(size_t)e * tv.tr_max + tr] = (int32_t)reached;
              tv.tr_time[(size_t)e * tv.tr_max + tr] = t_hop;
            }
            ++tr;
          }
          ++done;
          if (SAMPLE) records();
        }
      }
    }
    if (COUNT && l < done) {
      const uint32_t line = c.my_W & TGT_LINE_MASK, off = line - win_base;
      if (off < win_lines) atomicAdd(win + off, 1u);
      else atomicAdd(cbase + count_slot(line, v.count_stride), 1u);
    }
    if (done > 0u) {
      const uint4 r0 = s->reached[g][done - 1u][0], r1 = s->reached[g][done - 1u][1];
      n = r0.x;
      site = r0.y;
      gamma = __hiloint2double((int)r0.w, (int)r0.z);
      px = __uint_as_float(r1.x);
      py = __uint_as_float(r1.y);
      pz = __uint_as_float(r1.z);
    }
    h += done;
    active = active && done == most && h < h_end && t <= t_max && !trapped(n, gamma);
    wave_lds_fence();
  }
  if (v.live) {
    // excitons that a further launch could move (the budget aside)
    const uint64_t due = __ballot(valid && l == 0u && t <= t_max), b = due & __ballot(!trapped(n, gamma));
    // 8,192 waves ending together, one after another on one word, took 80 us of a launch
    if (lane == 0u) add_live(v.live + (blockIdx.x % LIVE_SLOTS) * LIVE_STRIDE, b, due);
  }
  if (!valid || l != 0u) return;
  v.x.site[e] = (int32_t)site;
  v.x.t_next[e] = t;
  v.x.hops[e] = h;
  v.x.dx[e] = dx;
  v.x.dy[e] = dy;
  v.x.dz[e] = dz;
  v.x.drains[e] = nd;
  v.x.hash[e] = hs;
  if (SAMPLE) v.x.k_rec[e] = k;
  if (TRACE && e < tv.n_trace) tv.tr_n[e] = tr;
}

// Positions as in k_hop, blockDim.x / 16 excitons to a workgroup; the workgroups of an XCD take its
// eighth of the order.  The departure counts of the lines around the workgroup's first exciton go
// to a window of 32-bit LDS counters (a launch's hops cannot wrap one: at most 2^32 departures per
// copy), the others to the XCD's copy.
constexpr uint32_t WIN_AHEAD = 8;  // 16-byte pieces of the window that a thread clears or reads at once

template <bool COUNT, bool SAMPLE, bool TRACE>
__global__ __launch_bounds__(256, 4) void k_hop_rows(hop_args a) {
  extern __shared__ uint4 rows_lds[];
  const uint32_t waves = blockDim.x >> 6, per_group = blockDim.x >> 4;
  batch_lds* s = reinterpret_cast<batch_lds*>(rows_lds) +
                 __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t* win = reinterpret_cast<uint32_t*>(reinterpret_cast<batch_lds*>(rows_lds) + waves);
  const uint32_t n = a.n_alive ? *a.n_alive : (uint32_t)a.v.x.n;
  const uint32_t groups = (n + per_group - 1u) / per_group;
  const uint32_t per_xcd = (groups + KMC_COUNT_COPIES - 1u) / KMC_COUNT_COPIES;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t quads = (a.win_lines + 3u) / 4u;  // of the window, in whole 16 bytes
  const uint32_t rank = blockIdx.x / KMC_COUNT_COPIES;
  const uint32_t p0 = ((blockIdx.x % KMC_COUNT_COPIES) * per_xcd + rank) * per_group;
  if (rank >= per_xcd || p0 >= n) return;
  const uint32_t pos = p0 + (threadIdx.x >> 4);
  const bool valid = pos < n;
  const uint32_t e = valid ? (a.perm ? a.perm[pos] : pos) : 0u;
  uint32_t base = 0u;
  if constexpr (COUNT) {
    for (uint32_t i = threadIdx.x; i < quads; i += WIN_AHEAD * blockDim.x)
#pragma unroll
      for (uint32_t k = 0; k < WIN_AHEAD; ++k)
        reinterpret_cast<uint4*>(win)[min(i + k * blockDim.x, quads - 1u)] = make_uint4(0u, 0u, 0u, 0u);
    if (a.win_lines < a.n_lines) {
      const uint32_t L0 = (uint32_t)a.v.roff[a.v.x.site[a.perm ? a.perm[p0] : p0]];
      base = L0 > a.win_lines / 2u ? L0 - a.win_lines / 2u : 0u;
      base = min(base, a.n_lines - a.win_lines);
    }
    __syncthreads();
  }
  hop_rows<COUNT, SAMPLE, TRACE>(a.v, e, valid, a.hop_budget, a.t_max, a.tv, s, lane, win, base,
                                 a.win_lines);
  if constexpr (COUNT) {
    __syncthreads();
    uint32_t* cbase = a.v.site_count + (size_t)xcd_id() * a.v.count_stride;
    for (uint32_t i = threadIdx.x; i < quads; i += WIN_AHEAD * blockDim.x) {
      uint4 q[WIN_AHEAD];
      uint32_t any = 0u;
#pragma unroll
      for (uint32_t k = 0; k < WIN_AHEAD; ++k) {
        q[k] = reinterpret_cast<const uint4*>(win)[min(i + k * blockDim.x, quads - 1u)];
        any |= q[k].x | q[k].y | q[k].z | q[k].w;
      }
      if (any == 0u) continue;
#pragma unroll
      for (uint32_t k = 0; k < WIN_AHEAD; ++k) {
        const uint32_t at = i + k * blockDim.x, cnt[4] = {q[k].x, q[k].y, q[k].z, q[k].w};
        if (at >= quads) break;
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
          if (cnt[j]) atomicAdd(cbase + count_slot(base + 4u * at + j, a.v.count_stride), cnt[j]);
      }
    }
  }
}

// The same with drift along the tubes (v > 0).
template <bool COUNT, bool SAMPLE, bool TRACE>
__global__ __launch_bounds__(256, 2) void k_hop_fly(hop_args a) {
  __shared__ uint4 rows[4 * 64 * ROW_UNITS];  // 8 KB of staged rows per wave
  __shared__ uint32_t win[COUNT_WINDOW_WORDS]; // 8 KB: the workgroup's departure-count window
  const uint32_t pos = xcd_position(), lane = threadIdx.x & 63u, n = (uint32_t)a.v.x.n;
  const bool valid = pos < n;
  const bool wave_live = __builtin_amdgcn_readfirstlane(pos - lane) < n;
  const uint32_t e = valid ? (a.perm ? a.perm[pos] : pos) : 0u;
  uint4* lds_wave = rows + 64u * ROW_UNITS * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  __shared__ net_view cold;
  if (threadIdx.x == 0) cold = a.v;
  uint32_t base = 0u;
  if constexpr (COUNT) {
    for (uint32_t i = threadIdx.x; i < COUNT_WINDOW_WORDS; i += blockDim.x) win[i] = 0u;
    const uint32_t p0 = pos - threadIdx.x;
    if (p0 < n) {
      const uint32_t L0 = (uint32_t)a.v.roff[a.v.x.site[a.perm ? a.perm[p0] : p0]];
      base = L0 > COUNT_WINDOW_LINES / 2 ? L0 - COUNT_WINDOW_LINES / 2 : 0u;
    }
  }
  __syncthreads();
  if (wave_live)
    hop_wave_fly<COUNT, SAMPLE, TRACE>(a.v, e, valid, a.hop_budget, a.t_max, a.tv, lds_wave, lane, win,
                                       base, cold);
  if constexpr (COUNT) {
    __syncthreads();
    window_flush(win, base, a.v.site_count + (size_t)xcd_id() * a.v.count_stride,
                 a.v.count_stride);
  }
}

// Several networks in one launch.  Network k's sorted excitons occupy positions
// [pbase[k], pbase[k] + n_k) of a position space whose network ranges start on workgroup
// boundaries, so every workgroup belongs to one network and reads that network's view with
// scalar loads; sorted entries of network k sit at [ebase[k], ebase[k] + n_k) of perm, which
// holds ensemble-wide exciton numbers ebase[k] + local id.  Departures are counted as in k_hop:
// an LDS window over the block lines around the workgroup's first exciton, flushed into that
// network's counts.
template <bool COUNT, bool SAMPLE>
__global__ __launch_bounds__(256, 4) void k_hop_ens(ens_args a) {
  __shared__ uint4 rows[4 * 64 * ROW_UNITS];  // 8 KB of staged rows per wave
  __shared__ uint32_t win[COUNT_WINDOW_WORDS]; // 8 KB: the workgroup's departure-count window
  const uint32_t pos = xcd_position();
  const uint32_t p0 = pos - threadIdx.x;       // the workgroup's first position
  if (p0 >= a.n_positions) return;             // the whole workgroup is past the end
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t net = __builtin_amdgcn_readfirstlane(a.wave_net[p0 >> 6]);
  const net_view v = a.nets[net];
  const int64_t q = (int64_t)pos - a.pbase[net];
  const bool valid = q < v.x.n;
  const bool wave_live = __builtin_amdgcn_readfirstlane((uint32_t)(q - lane < v.x.n));
  const int64_t eb = a.ebase[net];
  const uint32_t e = valid ? (uint32_t)((int64_t)a.perm[eb + q] - eb) : 0u;
  uint4* lds_wave = rows + 64u * ROW_UNITS * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if constexpr (!COUNT) {
    if (wave_live)
      hop_wave<COUNT, SAMPLE, false>(v, e, valid, a.hop_budget, a.t_max, trace_view{}, lds_wave,
                                     lane, nullptr, 0u);
  } else {
    for (uint32_t i = threadIdx.x; i < COUNT_WINDOW_WORDS; i += blockDim.x) win[i] = 0u;
    const int64_t q0 = (int64_t)p0 - a.pbase[net];
    uint32_t base = 0u;
    if (q0 < v.x.n) {
      const uint32_t e0 = (uint32_t)((int64_t)a.perm[eb + q0] - eb);
      const uint32_t L0 = (uint32_t)v.roff[v.x.site[e0]];
      base = L0 > COUNT_WINDOW_LINES / 2 ? L0 - COUNT_WINDOW_LINES / 2 : 0u;
    }
    __syncthreads();
    if (wave_live)
      hop_wave<COUNT, SAMPLE, false>(v, e, valid, a.hop_budget, a.t_max, trace_view{}, lds_wave,
                                     lane, win, base);
    __syncthreads();
    window_flush(win, base, v.site_count + (size_t)xcd_id() * v.count_stride, v.count_stride);
  }
}

hipError_t launch_hop_ens(const ens_args& a, bool count, bool sample, hipStream_t st) {
  const uint64_t groups = (a.n_positions + 255) / 256;
  const dim3 grid((unsigned)((groups + KMC_COUNT_COPIES - 1) / KMC_COUNT_COPIES * KMC_COUNT_COPIES)),
      block(256);
  if (count && sample) hipLaunchKernelGGL((k_hop_ens<true, true>), grid, block, 0, st, a);
  else if (count) hipLaunchKernelGGL((k_hop_ens<true, false>), grid, block, 0, st, a);
  else if (sample) hipLaunchKernelGGL((k_hop_ens<false, true>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((k_hop_ens<false, false>), grid, block, 0, st, a);
  return hipGetLastError();
}

// Sort keys of an ensemble's excitons: (network << 32) | first line of the current site's block.
__global__ __launch_bounds__(256) void k_ens_keys(int64_t n, const net_view* __restrict__ nets,
                                                  const uint16_t* __restrict__ exc_net,
                                                  const int64_t* __restrict__ ebase,
                                                  uint64_t* __restrict__ keys,
                                                  uint32_t* __restrict__ ids,
                                                  uint32_t* __restrict__ live) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g == 0 && live) live[0] = live[1] = 0u;
  if (g >= n) return;
  const uint32_t k = exc_net[g];
  const net_view& v = nets[k];
  const int64_t e = g - ebase[k];
  keys[g] = ((uint64_t)k << 32) | (uint64_t)(uint32_t)v.roff[v.x.site[e]];
  ids[g] = (uint32_t)g;
}

hipError_t launch_ens_keys(int64_t n, const net_view* nets, const uint16_t* exc_net,
                           const int64_t* ebase, uint64_t* keys, uint32_t* ids, uint32_t* live,
                           hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_ens_keys, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, nets,
                     exc_net, ebase, keys, ids, live);
  return hipGetLastError();
}

hipError_t launch_hop(const hop_args& a, bool count, bool sample, bool trace, bool fly,
                      hipStream_t st) {
  // a multiple of KMC_COUNT_COPIES workgroups, so the per-XCD chunks tile the excitons exactly
  const uint64_t groups = (a.v.x.n + 255) / 256;
  const dim3 grid((unsigned)((groups + KMC_COUNT_COPIES - 1) / KMC_COUNT_COPIES * KMC_COUNT_COPIES)),
      block(256);
#define KMC_HOP_CASE(C, S, T)                                            \
  if (count == C && sample == S && trace == T) {                         \
    if (fly) hipLaunchKernelGGL((k_hop_fly<C, S, T>), grid, block, 0, st, a); \
    else hipLaunchKernelGGL((k_hop<C, S, T>), grid, block, 0, st, a);    \
    return hipGetLastError();                                            \
  }
  KMC_HOP_CASE(false, false, false)
  KMC_HOP_CASE(true, false, false)
  KMC_HOP_CASE(false, true, false)
  KMC_HOP_CASE(true, true, false)
  KMC_HOP_CASE(false, false, true)
  KMC_HOP_CASE(true, false, true)
  KMC_HOP_CASE(false, true, true)
  KMC_HOP_CASE(true, true, true)
#undef KMC_HOP_CASE
  return hipErrorInvalidValue;
}

constexpr int64_t CU_LDS = 160 * 1024;

// A row of lanes per exciton pays up to 128 excitons per CU, two rounds of its waves: 1,250 hops with
// counts on 76,543 sites take 0.57 / 0.84 / 1.42 / 1.81 ms at 1,000 / 16,384 / 24,576 / 32,768
// excitons, k_hop's lane per exciton 1.86 / 1.92 / 1.96 / 1.94 ms; at 32,768 on 5,000 sites 1.75 and
// 2.05, on 50,000 1.74 and 1.94, on 624,739 1.79 and 2.12.
bool hop_rows_pays(int64_t walked, int n_cu) { return walked <= (int64_t)128 * n_cu; }

hipError_t launch_hop_rows(hop_args a, int64_t walked, uint32_t n_lines, int n_cu, bool count,
                           bool sample, bool trace, hipStream_t st) {
  int bs = 64;
  while (bs < 256 && walked * 16 > (int64_t)bs * n_cu) bs *= 2;
  const int64_t groups = (walked * 16 + bs - 1) / bs;
  const int64_t grid = (groups + KMC_COUNT_COPIES - 1) / KMC_COUNT_COPIES * KMC_COUNT_COPIES;
  // the window takes what the workgroups that share a CU leave of its LDS, but no more than a
  // launch's hops pay for: a thread clears and flushes four lines at a time, one such turn per hop
  // and 16 at most (one hop of one exciton on 300,000 sites: 56 us of clearing and flushing 39,000
  // lines by a single wave, as against a hop kernel of 5; 1,000 excitons' 2,500 hops there 1.69 ms
  // with 4,096 lines for that wave, 1.86 with 39,000)
  const int64_t paid = 4 * (int64_t)std::min<uint64_t>(a.hop_budget, 16u) * bs;
  const int64_t share = CU_LDS / std::max<int64_t>(1, std::min<int64_t>(8, (grid + n_cu - 1) / n_cu)) - 1024;
  const int64_t batches = (int64_t)(bs / 64) * (int64_t)sizeof(batch_lds);
  a.n_lines = n_lines;
  const int64_t fits = std::max<int64_t>(0, (share - batches) / 16 * 4);
  a.win_lines = count ? (uint32_t)std::min<int64_t>({n_lines, fits, paid}) : 0u;
  const size_t lds = (size_t)(batches + 16ll * ((a.win_lines + 3) / 4));
#define KMC_ROWS_CASE(C, S, T)                                                                 \
  if (count == C && sample == S && trace == T) {                                               \
    hipLaunchKernelGGL((k_hop_rows<C, S, T>), dim3((unsigned)grid), dim3(bs), lds, st, a);     \
    return hipGetLastError();                                                                  \
  }
  KMC_ROWS_CASE(false, false, false)
  KMC_ROWS_CASE(true, false, false)
  KMC_ROWS_CASE(false, true, false)
  KMC_ROWS_CASE(true, true, false)
  KMC_ROWS_CASE(false, false, true)
  KMC_ROWS_CASE(true, false, true)
  KMC_ROWS_CASE(false, true, true)
  KMC_ROWS_CASE(true, true, true)
#undef KMC_ROWS_CASE
  return hipErrorInvalidValue;
}

// The per-XCD copies of the departure counts folded into the 64-bit per-site totals and zeroed.
// Thread q owns block line q (slots and lines correspond one to one) in all copies; only a
// block's first line is ever counted, and its header gives the site.
__global__ __launch_bounds__(256) void k_fold_counts(int64_t n_lines, int64_t stride,
                                                     const uint4* __restrict__ blocks,
                                                     uint32_t* __restrict__ copies,
                                                     uint64_t* __restrict__ totals) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n_lines) return;
  uint64_t s = 0;
  const uint32_t slot = count_slot((uint32_t)q, stride);
#pragma unroll
  for (int x = 0; x < KMC_COUNT_COPIES; ++x) {
    uint32_t* c = copies + (size_t)x * stride + slot;
    const uint32_t v = *c;
    if (v) {
      s += v;
      *c = 0u;
    }
  }
  if (s) totals[blocks[(size_t)ROW_UNITS * q].y] += s;
}

// =============================================================================================
// (d) MSD / current reduction: block (k, b) reduces bin k over exciton batch b in a fixed
//     order (per-thread strided sums, wavefront shuffle tree, LDS across waves).  Bound by memory,
//     with a workgroup per bin and batch: in large batches each thread has the records of eight
//     excitons in flight (16 M excitons, 8 bins, 32 batches: 0.60 ms, 2.36 with one).
// =============================================================================================
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

// AHEAD > 1: records in flight together, read before it is known which excitons have reached the bin
// -- unless none of the wave's last AHEAD x 64 had.
template <int AHEAD>
__global__ __launch_bounds__(256) void k_reduce_samples(reduce_args a) {
  __shared__ double lds[5][4];
  const int k = blockIdx.x, b = blockIdx.y;
  const int64_t E = a.n_exc;
  const int64_t e0 = (int64_t)b * E / a.n_batches, e1 = (int64_t)(b + 1) * E / a.n_batches;
  double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  const uint32_t bin = (uint32_t)(a.bin0 + k);
  bool look = true;
  for (int64_t base = e0 + threadIdx.x; base < e1; base += AHEAD * blockDim.x) {
    if constexpr (AHEAD == 1) {
      if (bin < a.k_rec[base]) {
        const size_t r = (size_t)k * E + base;
        const double x = a.rec_dx[r], y = a.rec_dy[r], z = a.rec_dz[r];
        acc[0] += 1.0;
        acc[1] += x * x;
        acc[2] += y * y;
        acc[3] += z * z;
        acc[4] += (double)a.rec_drain[r];
      }
    } else {
      double x[AHEAD], y[AHEAD], z[AHEAD];
      uint32_t n[AHEAD], nd[AHEAD];
      const auto at = [&](int i) { return base + i * blockDim.x < e1 ? base + i * blockDim.x : base; };
      bool any = false;
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) n[i] = a.k_rec[at(i)];
      if (look) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) any |= bin < n[i];
        if (__ballot(any) == 0ull) continue;
      }
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) {
        const size_t r = (size_t)k * E + at(i);
        x[i] = a.rec_dx[r];
        y[i] = a.rec_dy[r];
        z[i] = a.rec_dz[r];
        nd[i] = a.rec_drain[r];
      }
      any = false;
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) {
        any |= bin < n[i];
        if (base + i * blockDim.x < e1 && bin < n[i]) {
          acc[0] += 1.0;
          acc[1] += x[i] * x[i];
          acc[2] += y[i] * y[i];
          acc[3] += z[i] * z[i];
          acc[4] += (double)nd[i];
        }
      }
      look = __ballot(any) == 0ull;
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    const double v = wave_sum(acc[q]);
    if (lane == 0) lds[q][wave] = v;
  }
  __syncthreads();
  if (threadIdx.x < 5) {
    const int q = threadIdx.x;
    const double v = (lds[q][0] + lds[q][1]) + (lds[q][2] + lds[q][3]);
    a.out[((size_t)k * a.n_batches + b) * 5 + q] = v;
  }
}

// Records in flight pay from a group of them per thread on: 64 bins of 1 M excitons in 100 batches
// take 0.30 ms, 0.34 with one at a time, in 1,000 batches 0.37 and 0.34.
hipError_t launch_reduce(const reduce_args& a, hipStream_t st) {
  const dim3 grid(a.n_bins, a.n_batches);
  if (a.n_exc / a.n_batches >= 8 * 256)
    hipLaunchKernelGGL(k_reduce_samples<8>, grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL(k_reduce_samples<1>, grid, dim3(256), 0, st, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// launch wrappers for (a) and (b)
// ---------------------------------------------------------------------------------------------
// =============================================================================================
// Contact (steady-state) mode: monte_carlo::step, save_population_profile,
// save_currents and repopulate_contacts (src/monte_carlo/monte_carlo.h:343-355, 443-516, 525-630).
// A particle's draws are keyed by its id (unique over the run) and its own hop count, so slots
// can be compacted and reused without any draw repeating.
// =============================================================================================
__device__ __forceinline__ int contact_section(double y, double ymin, double dy, int n_seg) {
#pragma clang fp contract(off)
  // save_population_profile (monte_carlo.h:567-568): truncation toward zero, then clamped
  int i = (int)((y - ymin) / dy);
  return i < 0 ? 0 : (i < n_seg ? i : n_seg - 1);
}

// The population and crossing counts of one particle's step (save_population_profile,
// save_currents: monte_carlo.h:565-571, 598-626) into the workgroup's LDS counters.  Interface k
// lies at ymin + dy (k + 1); +1 for a crossing upward (old < y_k <= new), -1 downward.
// Interfaces more than one section away from both positions cannot lie between them, so only
// those near the two sections are compared.
__device__ __forceinline__ void contact_tally(const contact_args& a, double y_old, double y_new,
                                              int32_t* s_pop, int32_t* s_cur) {
#pragma clang fp contract(off)
  const int i_new = contact_section(y_new, a.ymin, a.dy, a.n_seg);
  atomicAdd(&s_pop[i_new], 1);
  if (y_old != y_new) {
    const int i_old = contact_section(y_old, a.ymin, a.dy, a.n_seg);
    const int k_lo = max(0, min(i_old, i_new) - 1);
    const int k_hi = min(a.n_seg - 2, max(i_old, i_new) + 1);
    for (int k = k_lo; k <= k_hi; ++k) {
      const double yk = a.ymin + a.dy * (double)(k + 1);
      if (y_old < yk && y_new >= yk) atomicAdd(&s_cur[k], 1);
      else if (y_old >= yk && y_new < yk) atomicAdd(&s_cur[k], -1);
    }
  }
}

// particle::step (src/monte_carlo/particle.cpp:57-80) over one step with drift (v > 0), one
// thread per particle: the flight up to each due hop, the hop from the site reached, then the
// flight to the step's end, which is taken (particle::fly(dt), particle.cpp:77) and leaves the
// particle between sites.
__global__ __launch_bounds__(256) void k_contact_fly(contact_args a) {
#pragma clang fp contract(off)
  __shared__ int32_t s_pop[CONTACT_MAX_SEG], s_cur[CONTACT_MAX_SEG];
  __shared__ unsigned long long s_made;
  for (int i = threadIdx.x; i < a.n_seg; i += blockDim.x) s_pop[i] = s_cur[i] = 0;
  if (threadIdx.x == 0) s_made = 0ull;
  __syncthreads();
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < *a.n_live) {
    // slots in the order of their sites' rows: neighbouring lanes read neighbouring rows
    const int64_t e = a.perm ? (int64_t)a.perm[j] : j;
    const uint32_t id = a.s.id[e];
    double t = a.s.t_next[e];
    uint64_t h = a.s.hops[e];
    const uint32_t L0 = (uint32_t)a.roff[a.s.site[e]];
    uint32_t R = row_word(L0, a.blocks[(size_t)ROW_UNITS * L0].x);
    row_regs row = load_row(a.blocks, R);
    const double y_old = a.s.y[e];
    double tl = a.s.t_last[e];
    flight_state g{R, row.site, row.x, row.y, row.z, a.s.s_off[e], (uint32_t)a.s.heading[e],
                   0.0, 0.0, 0.0, 0u, 0ull};
    fly_leg leg = load_leg(a.fv, R, g.heading);
    uint64_t made = 0;
    hop_words hw;
    while (t <= a.t_end) {
      if (!fly(a.fv, g, leg, t - tl, id, h)) {
        atomicOr(a.err, CONTACT_ERR_FLY);
        break;
      }
      if (g.R != R) {
        R = g.R;
        row = load_row(a.blocks, R);
      }
      if (trapped(row.n, row.gamma)) {
        // no rates: the particle stays on its tube and flies on (scatterer.cpp:14-15)
        tl = t;
        t = INFINITY;
        ++h;
        break;
      }
      if (made == a.max_hops) {
        atomicOr(a.err, CONTACT_ERR_HOPS);
        break;
      }
      uint32_t w_sel, w_dw;
      hw.get(a.seed, id, h, w_sel, w_dw);
      const double dice = div_rand_max(row.gamma * (double)r31(w_sel));
      const uint32_t idx = select_entry(a.blocks, R, row.c, row.n, dice);
      R = target_of(a.blocks, R, row, idx) & ~EDGE_DRAIN_BIT;
      row = load_row(a.blocks, R);
      const uint32_t r = nonzero_draw1(w_dw, a.seed, id, h, STREAM_HOP_REDRAW);
      g = flight_state{R, row.site, row.x, row.y, row.z, 0.0, g.heading, 0.0, 0.0, 0.0, 0u, 0ull};
      leg = load_leg(a.fv, R, g.heading);  // in flight while the dwell is drawn
      tl = t;
      t = t + dwell_time(row.n, row.gamma, r);
      ++h;
      ++made;
    }
    if (!fly(a.fv, g, leg, a.t_end - tl, id, h)) atomicOr(a.err, CONTACT_ERR_FLY);
    tl = a.t_end;
    double ox, oy, oz;
    fly_offset(a.fv, g, leg, ox, oy, oz);
    const double y_new = a.py[g.site] + oy;
    a.s.site[e] = (int32_t)g.site;
    a.s.heading[e] = (uint8_t)g.heading;
    a.s.s_off[e] = g.s;
    a.s.t_last[e] = tl;
    a.s.t_next[e] = t;
    a.s.hops[e] = h;
    a.s.y[e] = y_new;
    if (made) atomicAdd(&s_made, (unsigned long long)made);
    contact_tally(a, y_old, y_new, s_pop, s_cur);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < a.n_seg; i += blockDim.x) {
    if (s_pop[i]) atomicAdd(a.pop + i, s_pop[i]);
    if (i + 1 < a.n_seg && s_cur[i]) atomicAdd(a.cur + i, s_cur[i]);
  }
  if (threadIdx.x == 0 && s_made) atomicAdd(a.hops_made, s_made);
}

// The order in which a step takes the live slots: by contact_key, ORDER_BINS values, in two
// launches over tiles of SCAN_TILE slots.  k_contact_keys counts every key's slots, k_contact_order
// gives each tile its places behind the counts of the keys below.  Slots of one key stand in no
// particular order (it changes no result).  At 1 M slots the pair takes 35 us, a library radix sort
// of the same 8-bit keys with their kernel 75; at 52,000 slots 15 us for 43 (seven launches).
__global__ __launch_bounds__(SCAN_THREADS) void k_contact_keys(const int64_t* n_live,
                                                               const int32_t* __restrict__ site,
                                                               const int64_t* __restrict__ roff,
                                                               const uint8_t* __restrict__ chir,
                                                               contact_key_layout kl,
                                                               contact_order o) {
  __shared__ uint32_t cnt[ORDER_BINS];
  cnt[threadIdx.x] = 0u;
  __syncthreads();
  const int64_t n = *n_live, base = (int64_t)blockIdx.x * SCAN_TILE + threadIdx.x;
#pragma unroll
  for (int i = 0; i < SCAN_ITEMS; ++i) {
    const int64_t e = base + i * SCAN_THREADS;
    if (e >= n) continue;
    const int32_t s = site[e];
    const uint32_t row = (uint32_t)roff[s];
    const uint32_t region = (uint32_t)((uint64_t)row * KMC_COUNT_COPIES / kl.lines);
    const uint32_t first = (uint32_t)(((uint64_t)region * kl.lines) / KMC_COUNT_COPIES);
    const uint32_t k = (region << (kl.chir_bits + kl.row_bits)) |
                       ((uint32_t)chir[s] << kl.row_bits) |
                       ((row - first) >> kl.row_shift);
    o.key[e] = (uint8_t)k;
    atomicAdd(&cnt[k], 1u);
  }
  __syncthreads();
  if (cnt[threadIdx.x]) atomicAdd(o.count + threadIdx.x, cnt[threadIdx.x]);
}

__global__ __launch_bounds__(SCAN_THREADS) void k_contact_order(const int64_t* n_live,
                                                                contact_order o) {
  __shared__ uint32_t cnt[ORDER_BINS], first[ORDER_BINS];
  __shared__ int64_t lds[SCAN_THREADS / 64];
  cnt[threadIdx.x] = 0u;
  __syncthreads();
  const int64_t n = *n_live, base = (int64_t)blockIdx.x * SCAN_TILE + threadIdx.x;
  uint32_t key[SCAN_ITEMS], rank[SCAN_ITEMS];
#pragma unroll
  for (int i = 0; i < SCAN_ITEMS; ++i) {
    const int64_t e = base + i * SCAN_THREADS;
    if (e >= n) continue;
    key[i] = o.key[e];
    rank[i] = atomicAdd(&cnt[key[i]], 1u);
  }
  __syncthreads();
  int64_t total;
  const int64_t below = block_exclusive_scan(o.count[threadIdx.x], lds, &total);
  const uint32_t mine = cnt[threadIdx.x];
  first[threadIdx.x] = (uint32_t)below + (mine ? atomicAdd(o.cursor + threadIdx.x, mine) : 0u);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < SCAN_ITEMS; ++i) {
    const int64_t e = base + i * SCAN_THREADS;
    if (e < n) o.perm[first[key[i]] + rank[i]] = (uint32_t)e;
  }
}

// particle::step of every live particle for v = 0, built like the Kubo kernel's wave loop around
// the cooperative row load: every lane of a wave takes part in every row load, and the wave
// loops until no lane has a hop due by the step's end (a lane whose particle has stopped keeps
// taking part in the loads).  The next hop is selected as soon as a row arrives and its row load issued
// before the dwell at the current site is drawn and the clock tested, so the load is in flight
// meanwhile.  Each particle's arithmetic and its order are those of the oracle's step.  The live
// slots, sorted by region, chirality and row, are dealt to the XCDs in eighths (from the
// device-side live count), so each XCD's L2 serves one compact region of the film.  The grid is
// a multiple of 8 workgroups covering the capacity.
__global__ __launch_bounds__(256, 4) void k_contact_wave(contact_args a) {
#pragma clang fp contract(off)
  __shared__ uint4 rows[4 * 64 * ROW_UNITS];  // 8 KB of staged rows per wave
  __shared__ unsigned long long s_made;
  // the section counters are sized by the launch (2 n_seg words), so that four workgroups fit
  // a CU's LDS beside the staged rows
  extern __shared__ int32_t s_counts[];
  int32_t* s_pop = s_counts;
  int32_t* s_cur = s_counts + a.n_seg;
  for (int i = threadIdx.x; i < a.n_seg; i += blockDim.x) s_pop[i] = s_cur[i] = 0;
  if (threadIdx.x == 0) s_made = 0ull;
  __syncthreads();
  const int64_t n_live = *a.n_live;
  const uint32_t groups = (uint32_t)((n_live + 255) / 256);
  const uint32_t per_xcd = (groups + KMC_COUNT_COPIES - 1) / KMC_COUNT_COPIES;
  const uint32_t b = blockIdx.x;
  const int64_t j = (b / KMC_COUNT_COPIES < per_xcd)
                        ? ((int64_t)((b % KMC_COUNT_COPIES) * per_xcd + b / KMC_COUNT_COPIES) * 256 +
                           threadIdx.x)
                        : INT64_MAX;
  const bool valid = j < n_live;
  const uint32_t lane = threadIdx.x & 63u;
  if (__ballot(valid) != 0) {
    uint4* lds_wave = rows + 64u * ROW_UNITS * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t e = valid ? (a.perm ? (int64_t)a.perm[j] : j) : 0;
    uint32_t id = 0, W = 0, r_dw = 0;
    double t = INFINITY, y_old = 0.0;
    uint64_t h = 0, made = 0;
    if (valid) {
      id = a.s.id[e];
      t = a.s.t_next[e];
      h = a.s.hops[e];
      y_old = a.s.y[e];
      const uint32_t L0 = (uint32_t)a.roff[a.s.site[e]];
      W = row_word(L0, a.blocks[(size_t)ROW_UNITS * L0].x);
    }
    bool active = valid, pend = false;
    uint32_t site_now = 0;  // when stopped: the site it stopped at (the row loaded after that
                            // may be the one of the hop selected but not made)
    hop_words hw;
    coop_issue(a.blocks, W, lds_wave, lane);
    while (true) {
      __builtin_amdgcn_s_setprio(2);  // raised until the next row load is out, as in hop_wave
      const coop_row row = coop_finish(lds_wave, lane);
      // (A) the hop from this site, selected before the clock test that decides whether it is
      // made, and the load of the row it leads to, in flight while (B) and (C) run
      const bool can = active && !trapped(row.n, row.gamma) && made < a.max_hops;
      uint32_t W_next = W, r_next = 0;
      if (can) {
        uint32_t w_sel, w_dw;
        hw.get(a.seed, id, h, w_sel, w_dw);
        const double dice = div_rand_max(row.gamma * (double)r31(w_sel));
        const uint32_t idx = select_entry(a.blocks, W, row.c, row.n, dice);
        const uint32_t tg = idx < ROW_INLINE ? target_lds(lds_wave, lane, idx)
                                             : target_wide(a.blocks, W, row.n, idx);
        W_next = tg & ~EDGE_DRAIN_BIT;
        r_next = nonzero_draw1(w_dw, a.seed, id, h, STREAM_HOP_REDRAW);
      }
      // a lane whose particle has stopped never reads its row again: it loads block line 0,
      // which every such lane of the wave shares, instead of its own row
      coop_issue(a.blocks, active ? W_next : 0u, lds_wave, lane);
      __builtin_amdgcn_s_setprio(0);
      // (B) the dwell at this site of the hop that led here
      if (pend) {
        t = t + dwell_time(row.n, row.gamma, r_dw);
        pend = false;
      }
      // (C) the hop of (A) is made if it falls due by the step's end
      if (active) {
        if (!(t <= a.t_end) || trapped(row.n, row.gamma)) {
          active = false;
        } else if (made == a.max_hops) {
          atomicOr(a.err, CONTACT_ERR_HOPS);
          active = false;
        }
        if (!active) site_now = row.site;
      }
      if (active) {
        W = W_next;
        r_dw = r_next;
        pend = true;
        ++h;
        ++made;
      }
      if (__ballot(active) == 0) break;
    }
    // the last issued load lands in this wave's LDS rows: wait for it before the wave moves on
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (valid) {
      const double y_new = a.py[site_now];
      a.s.site[e] = (int32_t)site_now;
      a.s.t_next[e] = t;
      a.s.hops[e] = h;
      a.s.y[e] = y_new;
      if (made) atomicAdd(&s_made, (unsigned long long)made);
      contact_tally(a, y_old, y_new, s_pop, s_cur);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < a.n_seg; i += blockDim.x) {
    if (s_pop[i]) atomicAdd(a.pop + i, s_pop[i]);
    if (i + 1 < a.n_seg && s_cur[i]) atomicAdd(a.cur + i, s_cur[i]);
  }
  if (threadIdx.x == 0 && s_made) atomicAdd(a.hops_made, s_made);
}

// repopulate (monte_carlo.h:461-474): a particle whose y lies in [y_lo, y_hi] leaves
__global__ __launch_bounds__(256) void k_contact_keep(contact_args a, int64_t n, double y_lo,
                                                      double y_hi, uint32_t* keep) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  uint32_t k = 0;
  if (e < *a.n_live) {
    const double y = a.s.y[e];
    k = (y >= y_lo && y <= y_hi) ? 0u : 1u;
  }
  keep[e] = k;
}

// The kept particles, in slot order, to the front of the other buffer.
__global__ __launch_bounds__(256) void k_contact_compact(int64_t capacity, contact_slots src,
                                                         contact_slots dst,
                                                         const uint32_t* __restrict__ keep,
                                                         const int64_t* __restrict__ off) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= capacity || !keep[e]) return;
  const int64_t o = off[e];
  dst.site[o] = src.site[e];
  dst.t_next[o] = src.t_next[e];
  dst.hops[o] = src.hops[e];
  dst.id[o] = src.id[e];
  dst.y[o] = src.y[e];
  dst.heading[o] = src.heading[e];
  dst.s_off[o] = src.s_off[e];
  dst.t_last[o] = src.t_last[e];
}

// A new particle in `slot` on a site of `sites`, as the particle constructor makes it
// (particle.h:49-52): a random site of the list (rand() % size), the first dwell from the site
// (ff_time), then the heading (rand() % 2).
__device__ __forceinline__ void contact_new(const contact_args& a, int64_t slot, uint64_t id64,
                                            const int32_t* __restrict__ sites, int64_t n_sites,
                                            double t_now) {
#pragma clang fp contract(off)
  if (slot >= a.capacity) {
    atomicOr(a.err, CONTACT_ERR_CAPACITY);
    return;
  }
  if (id64 > 0xFFFFFFFFull) {
    atomicOr(a.err, CONTACT_ERR_IDS);
    return;
  }
  const uint32_t id = (uint32_t)id64;
  const u32x4 w = draw4(a.seed, id, 0, STREAM_CONTACT);
  const int32_t site = sites[r31(w.v[0]) % (uint32_t)n_sites];
  const uint4 hh = a.blocks[(size_t)ROW_UNITS * a.roff[site]];
  const uint32_t r = nonzero_draw(w.v[1], w.v[3], a.seed, id, 0, STREAM_CONTACT_REDRAW);
  a.s.site[slot] = (int32_t)hh.y;
  a.s.t_next[slot] = t_now + dwell_time(hh.x, __hiloint2double((int)hh.w, (int)hh.z), r);
  a.s.hops[slot] = 0;
  a.s.id[slot] = id;
  a.s.y[slot] = a.py[site];
  a.s.heading[slot] = (uint8_t)(r31(w.v[2]) & 1u);
  a.s.s_off[slot] = 0.0;
  a.s.t_last[slot] = t_now;
}

// `count` new particles in slots *base + k; ids continue from *next_id.
__global__ __launch_bounds__(256) void k_contact_inject(contact_args a, const int64_t* base,
                                                        int64_t count,
                                                        const int32_t* __restrict__ sites,
                                                        int64_t n_sites,
                                                        const uint64_t* __restrict__ next_id,
                                                        double t_now) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < count) contact_new(a, *base + k, *next_id + (uint64_t)k, sites, n_sites, t_now);
}

__global__ void k_contact_finish(const int64_t* base, int64_t count, int64_t capacity,
                                 uint64_t* next_id, int64_t* n_live) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const int64_t n = *base + count;
  *n_live = n < capacity ? n : capacity;
  *next_id += (uint64_t)count;
}

// Repopulation of both contacts (monte_carlo.h:443-491) in three launches: contact 1 loses the
// particles whose y lies in its range and gets c_pop[0] new ones, then contact n_seg likewise; the
// kept particles keep their order and the new ones follow them, contact 1's first.  With disjoint
// ranges (checked by the caller) contact n_seg removes none of contact 1's new particles, so one
// pass over the slots decides for both.  Tiles of SCAN_TILE slots: k_contact_count counts what a
// tile keeps, k_contact_offsets scans the tiles, k_contact_move writes the other buffer.  The move
// is bound by memory: 72 bytes a particle read and written, by lanes on consecutive slots (eight
// consecutive slots to a lane, as in the scans: 72 us at 1 M particles, this way 16).  A pass per
// contact took fourteen launches; a step of 1 M particles took ~110 us outside its sort and step
// kernel, now 26.
__device__ __forceinline__ bool in_contact(const contact_move_args& m, int side, double y) {
  return y >= m.rm_lo[side] && y <= m.rm_hi[side];
}

__global__ __launch_bounds__(SCAN_THREADS) void k_contact_count(contact_move_args m) {
  __shared__ int32_t s_kept, s_first;
  if (threadIdx.x == 0) s_kept = s_first = 0;
  __syncthreads();
  const int64_t n = *m.n_live;
  const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + threadIdx.x;
  int32_t kept = 0, first = 0;  // kept by both contacts; by contact 1
#pragma unroll
  for (int i = 0; i < SCAN_ITEMS; ++i) {
    const int64_t e = base + i * SCAN_THREADS;
    const double y = e < n ? m.src.y[e] : 0.0;
    const bool k0 = e < n && !in_contact(m, 0, y);
    first += __popcll(__ballot(k0));
    kept += __popcll(__ballot(k0 && !in_contact(m, 1, y)));
  }
  if ((threadIdx.x & 63u) == 0) {
    atomicAdd(&s_kept, kept);
    atomicAdd(&s_first, first);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    m.tile_kept[blockIdx.x] = s_kept;
    m.tile_first[blockIdx.x] = s_first;
  }
}

__global__ __launch_bounds__(SCAN_THREADS) void k_contact_offsets(contact_move_args m, int64_t n_tiles) {
  __shared__ int64_t lds[SCAN_THREADS / 64];
  int64_t kept = 0, first = 0;
  for (int64_t base = 0; base < n_tiles; base += SCAN_THREADS) {
    const int64_t i = base + threadIdx.x;
    int64_t total;
    const int64_t ex = block_exclusive_scan(i < n_tiles ? m.tile_kept[i] : 0, lds, &total);
    if (i < n_tiles) m.tile_kept[i] = kept + ex;
    kept += total;
    (void)block_exclusive_scan(i < n_tiles ? m.tile_first[i] : 0, lds, &total);
    first += total;
  }
  m.order_count[threadIdx.x] = m.order_cursor[threadIdx.x] = 0u;  // for the next step's order
  if (threadIdx.x != 0) return;
  const int64_t live = kept + m.count[0] + m.count[1];
  if (first + m.count[0] > m.capacity || live > m.capacity) atomicOr(m.err, CONTACT_ERR_CAPACITY);
  m.base[0] = kept;
  m.base[1] = (int64_t)*m.next_id;
  m.base[2] = *m.n_live;  // the slots counted: k_contact_move looks at the same ones
  *m.next_id += (uint64_t)(m.count[0] + m.count[1]);
  *m.n_live = live < m.capacity ? live : m.capacity;
  *m.live_out = *m.n_live;
  *m.live_host = *m.n_live;  // pinned host memory
}

// Blocks [0, n_tiles): the kept particles; the rest: the new ones.
__global__ __launch_bounds__(SCAN_THREADS) void k_contact_move(contact_args a, contact_move_args m,
                                                               int64_t n_tiles) {
#pragma clang fp contract(off)
  __shared__ int32_t s_kept[SCAN_ITEMS * SCAN_THREADS / 64];
  if ((int64_t)blockIdx.x < n_tiles) {
    const int64_t n = m.base[2];
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint64_t keep[SCAN_ITEMS];
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
      const int64_t e = base + i * SCAN_THREADS;
      const double y = e < n ? m.src.y[e] : 0.0;
      keep[i] = __ballot(e < n && !in_contact(m, 0, y) && !in_contact(m, 1, y));
      if (lane == 0) s_kept[i * (SCAN_THREADS / 64) + wave] = __popcll(keep[i]);
    }
    __syncthreads();
    int64_t o = m.tile_kept[blockIdx.x];
    uint32_t before = 0;  // runs of 64 slots added to o
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
      for (; before < i * (SCAN_THREADS / 64) + wave; ++before) o += s_kept[before];
      if (!(keep[i] >> lane & 1u)) continue;
      const int64_t e = base + i * SCAN_THREADS;
      const int64_t to = o + __popcll(keep[i] & (((uint64_t)1 << lane) - 1u));
      m.dst.site[to] = m.src.site[e];
      m.dst.t_next[to] = m.src.t_next[e];
      m.dst.hops[to] = m.src.hops[e];
      m.dst.id[to] = m.src.id[e];
      m.dst.y[to] = m.src.y[e];
      if (m.drift) {
        m.dst.heading[to] = m.src.heading[e];
        m.dst.s_off[to] = m.src.s_off[e];
        m.dst.t_last[to] = m.src.t_last[e];
      }
    }
    return;
  }
  const int64_t k = ((int64_t)blockIdx.x - n_tiles) * blockDim.x + threadIdx.x;
  if (k >= m.count[0] + m.count[1]) return;
  const int side = k < m.count[0] ? 0 : 1;
  a.s = m.dst;
  contact_new(a, m.base[0] + k, (uint64_t)m.base[1] + (uint64_t)k, m.sites + m.list_off[side],
              m.list_n[side], m.t_now);
}

static inline dim3 grid_for(int64_t n) { return dim3((unsigned)((n + 255) / 256)); }

hipError_t launch_cell_assign(const site_arrays& s, const cell_desc& c, int32_t* cell_of,
                              uint32_t* cell_count, hipStream_t st) {
  if (s.n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_cell_assign, grid_for(s.n), dim3(256), 0, st, s, c, cell_of, cell_count);
  return hipGetLastError();
}

hipError_t launch_cell_scatter(int64_t n, const int32_t* cell_of, const int64_t* cell_start,
                               uint32_t* cell_fill, int32_t* cell_sites, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_cell_scatter, grid_for(n), dim3(256), 0, st, n, cell_of, cell_start,
                     cell_fill, cell_sites);
  return hipGetLastError();
}

hipError_t launch_cell_sort(int64_t n_cells, const int64_t* cell_start, int32_t* cell_sites,
                            hipStream_t st) {
  hipLaunchKernelGGL(k_cell_sort, grid_for(n_cells), dim3(256), 0, st, n_cells, cell_start,
                     cell_sites);
  return hipGetLastError();
}

// Sites of one launch of the pair search: its threads stay below 2^32.
constexpr int64_t STENCIL_SITES = (int64_t)1 << 26;
static dim3 stencil_grid(int64_t sites) {
  return grid_for(std::min(sites, STENCIL_SITES) * (int64_t)STENCIL_LANES);
}

hipError_t launch_count_pairs(const site_arrays& s, const cell_desc& c, const int64_t* cell_start,
                              const int32_t* cell_sites, uint32_t* deg, hipStream_t st) {
  if (s.n == 0) return hipSuccess;
  for (int64_t i0 = 0; i0 < s.n; i0 += STENCIL_SITES)
    hipLaunchKernelGGL(k_count_pairs, stencil_grid(s.n - i0), dim3(256), 0, st, i0, s, c,
                       cell_start, cell_sites, deg);
  return hipGetLastError();
}

hipError_t launch_fill_pairs(int mode, const site_arrays& s, const cell_desc& c,
                             const int64_t* cell_start, const int32_t* cell_sites,
                             const int64_t* row_ptr, int64_t nnz, const table_desc& t,
                             const csr_arrays& out, const pair_geom_arrays& geo, int32_t* err,
                             hipStream_t st) {
  if (s.n == 0) return hipSuccess;
  for (int64_t i0 = 0; i0 < s.n; i0 += STENCIL_SITES)
    hipLaunchKernelGGL(k_list_pairs, stencil_grid(s.n - i0), dim3(256), 0, st, i0, s, c, cell_start,
                       cell_sites, row_ptr, out);
  constexpr int64_t SLICE = (int64_t)1 << 30;
  for (int64_t p0 = 0; p0 < nnz; p0 += SLICE) {
    const dim3 grid = grid_for(std::min(nnz - p0, SLICE));
    if (mode == 0)
      hipLaunchKernelGGL(k_pair_values<0>, grid, dim3(256), 0, st, p0, nnz, s, c, t, out, geo);
    else
      hipLaunchKernelGGL(k_pair_values<1>, grid, dim3(256), 0, st, p0, nnz, s, c, t, out, geo);
  }
  const hipError_t e = hipGetLastError();
  return e != hipSuccess || mode != 0 ? e : launch_finish_pair_rates(s.n, out.cum, out, err, st);
}

hipError_t launch_unpack_edges(int64_t n, const edge_rec* edge, int32_t* col, float* disp,
                               hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_unpack_edges, grid_for(n), dim3(256), 0, st, n, edge, col, disp);
  return hipGetLastError();
}

hipError_t launch_unpack_rows(int64_t n, const site_hdr* hdr, int64_t* row, double* gamma,
                              hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_unpack_rows, grid_for(n), dim3(256), 0, st, n, hdr, row, gamma);
  return hipGetLastError();
}

// Zeroes several arrays in one launch, 16 bytes a lane.  A new run on a small film is a handful of
// arrays of a few kilobytes, where every launch costs ~4 us of host time and ~3 on the device
// (1,000 excitons on 5,000 sites: an injection 21 us with a memset per array, 17 with this; a
// sampling grid 23 and 13).
__global__ __launch_bounds__(256) void k_clear(clear_args a) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x, step = (size_t)gridDim.x * blockDim.x;
  for (int k = 0; k < a.n; ++k) {
    uint32_t* p = static_cast<uint32_t*>(a.p[k]);
    const size_t words = a.words[k], quads = words / 4;
    for (size_t i = t; i < quads; i += step)
      reinterpret_cast<uint4*>(p)[i] = make_uint4(0u, 0u, 0u, 0u);
    if (t < words % 4) p[4 * quads + t] = 0u;
  }
}

hipError_t launch_clear(const clear_args& a, hipStream_t st) {
  size_t most = 0;
  for (int k = 0; k < a.n; ++k) {
    if ((uintptr_t)a.p[k] % 16 != 0) return hipErrorInvalidValue;
    most = std::max(most, a.words[k]);
  }
  if (most == 0) return hipSuccess;
  // up to 4,096 workgroups: beyond them a lane takes several pieces
  const size_t groups = std::min<size_t>((most / 4 + 255) / 256 + 1, 4096);
  hipLaunchKernelGGL(k_clear, dim3((unsigned)groups), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_interleave3(int64_t n, const double* x, const double* y, const double* z,
                              double* out, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_interleave3, grid_for(n), dim3(256), 0, st, n, x, y, z, out);
  return hipGetLastError();
}

hipError_t launch_finish_pair_rates(int64_t n, const double* rates, const csr_arrays& out,
                                    int32_t* err, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_finish_pair_rates, grid_for(n), dim3(256), 0, st, n, rates, out, err);
  return hipGetLastError();
}

hipError_t launch_inject(const exciton_arrays& x, const uint4* blocks, const uint32_t* src_roff,
                         uint32_t n_src, uint64_t seed, hipStream_t st) {
  if (x.n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_inject, grid_for(x.n), dim3(256), 0, st, x, blocks, src_roff, n_src, seed);
  return hipGetLastError();
}

hipError_t launch_block_sizes(int64_t n, const site_hdr* hdr, const int32_t* order, uint32_t* lines,
                              hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_block_sizes, grid_for(n), dim3(256), 0, st, n, hdr, order, lines);
  return hipGetLastError();
}

hipError_t launch_place_blocks(int64_t n, const int32_t* order, const int64_t* first, int64_t* roff,
                               hipStream_t st) {
  hipLaunchKernelGGL(k_place_blocks, grid_for(n + 1), dim3(256), 0, st, n, order, first, roff);
  return hipGetLastError();
}

hipError_t launch_exciton_keys(int64_t n, const int32_t* site, const int64_t* roff,
                               const idle_test& it, uint32_t* keys, uint32_t* ids, uint32_t* live,
                               hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_exciton_keys, grid_for(n), dim3(256), 0, st, n, site, roff, it, keys, ids,
                     live);
  return hipGetLastError();
}

hipError_t launch_fill_blocks(int64_t n, const site_hdr* hdr, const double* cum,
                              const edge_rec* edge, const int64_t* roff, const double* px,
                              const double* py, const double* pz, uint4* blocks, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_pack_rows, grid_for(n), dim3(256), 0, st, n, hdr, cum, edge, roff, px, py,
                     pz, blocks);
  return hipGetLastError();
}

// Chirality class (donor * n_chir + acceptor) of every CSR entry, and per-class index lists.
// Class counts are summed per workgroup in LDS first (a film of one chirality puts every pair
// in one class), then one device atomic per class and workgroup.
constexpr int MAX_PAIR_CLASSES = 256;

__device__ __forceinline__ void clear_class_counts(uint32_t* lds) {
  for (int c = threadIdx.x; c < MAX_PAIR_CLASSES; c += blockDim.x) lds[c] = 0u;
  __syncthreads();
}

__device__ __forceinline__ void flush_class_counts(const uint32_t* lds, uint32_t* __restrict__ counts,
                                                   int n_classes) {
  __syncthreads();
  for (int c = threadIdx.x; c < n_classes; c += blockDim.x)
    if (lds[c]) atomicAdd(&counts[c], lds[c]);
}

__global__ __launch_bounds__(256) void k_pair_class(int64_t n, const site_hdr* __restrict__ hdr,
                                                    const edge_rec* __restrict__ edge,
                                                    const uint8_t* __restrict__ chir, int32_t n_chir,
                                                    uint8_t* __restrict__ cls,
                                                    uint32_t* __restrict__ counts) {
  __shared__ uint32_t lds[MAX_PAIR_CLASSES];
  clear_class_counts(lds);
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const site_hdr h = hdr[i];
    const int ci = chir[i];
    for (uint32_t k = 0; k < h.n; ++k) {
      const int cj = chir[edge[h.rs + k].col & EDGE_COL_MASK];
      const int c = ci * n_chir + cj;
      cls[h.rs + k] = (uint8_t)c;
      atomicAdd(&lds[c], 1u);
    }
  }
  flush_class_counts(lds, counts, n_chir * n_chir);
}

// entries with mask[p] == 0 (mask optional) are left out
// Slots within a class: a workgroup first numbers its own entries per class in LDS, then
// reserves one range per class with a single device atomic.
__global__ __launch_bounds__(256) void k_pair_scatter(int64_t nnz, const uint8_t* __restrict__ cls,
                                                      const uint8_t* __restrict__ mask,
                                                      const int64_t* __restrict__ starts,
                                                      uint32_t* __restrict__ fill,
                                                      int64_t* __restrict__ sel) {
  __shared__ uint32_t local[MAX_PAIR_CLASSES];
  __shared__ uint32_t base[MAX_PAIR_CLASSES];
  clear_class_counts(local);
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool take = p < nnz && (!mask || mask[p]);
  const int c = take ? (int)cls[p] : 0;
  const uint32_t slot = take ? atomicAdd(&local[c], 1u) : 0u;
  __syncthreads();
  for (int q = threadIdx.x; q < MAX_PAIR_CLASSES; q += blockDim.x)
    base[q] = local[q] ? atomicAdd(&fill[q], local[q]) : 0u;
  __syncthreads();
  if (take) sel[starts[c] + base[c] + slot] = p;
}

hipError_t launch_pair_classes(int64_t n, int64_t nnz, const site_hdr* hdr, const edge_rec* edge,
                               const uint8_t* chir, int32_t n_chir, uint8_t* cls, uint32_t* counts,
                               hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_pair_class, grid_for(n), dim3(256), 0, st, n, hdr, edge, chir, n_chir, cls,
                     counts);
  (void)nnz;
  return hipGetLastError();
}

hipError_t launch_pair_scatter(int64_t nnz, const uint8_t* cls, const uint8_t* mask,
                               const int64_t* starts, uint32_t* fill, int64_t* sel, hipStream_t st) {
  if (nnz == 0) return hipSuccess;
  hipLaunchKernelGGL(k_pair_scatter, grid_for(nnz), dim3(256), 0, st, nnz, cls, mask, starts, fill, sel);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_mask_count(int64_t nnz, const uint8_t* __restrict__ cls,
                                                    const uint8_t* __restrict__ mask,
                                                    uint32_t* __restrict__ counts) {
  __shared__ uint32_t lds[MAX_PAIR_CLASSES];
  clear_class_counts(lds);
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < nnz && mask[p]) atomicAdd(&lds[cls[p]], 1u);
  flush_class_counts(lds, counts, MAX_PAIR_CLASSES);
}

hipError_t launch_mask_count(int64_t nnz, const uint8_t* cls, const uint8_t* mask, uint32_t* counts,
                             hipStream_t st) {
  if (nnz == 0) return hipSuccess;
  hipLaunchKernelGGL(k_mask_count, grid_for(nnz), dim3(256), 0, st, nnz, cls, mask, counts);
  return hipGetLastError();
}

hipError_t launch_fly_table(int64_t n, const int32_t* left, const int32_t* right,
                            const uint8_t* flags, const int64_t* roff, const site_hdr* hdr,
                            const double* px, const double* py, const double* pz,
                            const double* half_per, uint4* table, int32_t* bad, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fly_table, grid_for(2 * n), dim3(256), 0, st, n, left, right, flags, roff, hdr,
                     px, py, pz, half_per[0], half_per[1], half_per[2], table, bad);
  return hipGetLastError();
}

hipError_t launch_morton_keys(int64_t n, const int32_t* cell_of, int32_t nx, int32_t ny,
                              uint64_t* keys, int32_t* ids, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_morton_keys, grid_for(n), dim3(256), 0, st, n, cell_of, nx, ny, keys, ids);
  return hipGetLastError();
}

hipError_t launch_gather_offsets(int64_t n, const int32_t* idx, const int64_t* roff,
                                 const site_hdr* hdr, uint32_t* out, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_gather_offsets, grid_for(n), dim3(256), 0, st, n, idx, roff, hdr, out);
  return hipGetLastError();
}

hipError_t launch_fold_counts(int64_t n_lines, int64_t stride, const uint4* blocks,
                              uint32_t* copies, uint64_t* totals, hipStream_t st) {
  if (n_lines == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fold_counts, grid_for(n_lines), dim3(256), 0, st, n_lines, stride, blocks,
                     copies, totals);
  return hipGetLastError();
}

hipError_t launch_contact_step(const contact_args& a, bool fly, int64_t n_max, hipStream_t st) {
  if (n_max == 0) return hipSuccess;
  if (a.n_seg < 1 || a.n_seg > CONTACT_MAX_SEG || n_max < 0 || n_max > a.capacity)
    return hipErrorInvalidValue;
  if (fly)
    hipLaunchKernelGGL(k_contact_fly, grid_for(n_max), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL(k_contact_wave,
                       dim3((unsigned)((n_max + 256 * KMC_COUNT_COPIES - 1) /
                                       (256 * KMC_COUNT_COPIES) * KMC_COUNT_COPIES)),
                       dim3(256), (size_t)2 * a.n_seg * sizeof(int32_t), st, a);
  return hipGetLastError();
}

hipError_t launch_contact_order(int64_t n, const int64_t* n_live, const int32_t* site,
                                const int64_t* roff, const uint8_t* chir,
                                const contact_key_layout& kl, const contact_order& o,
                                hipStream_t st) {
  static_assert(ORDER_BINS == SCAN_THREADS, "a thread per key");
  if (n == 0) return hipSuccess;
  const dim3 grid((unsigned)((n + SCAN_TILE - 1) / SCAN_TILE));
  hipLaunchKernelGGL(k_contact_keys, grid, dim3(SCAN_THREADS), 0, st, n_live, site, roff, chir, kl, o);
  hipLaunchKernelGGL(k_contact_order, grid, dim3(SCAN_THREADS), 0, st, n_live, o);
  return hipGetLastError();
}

hipError_t launch_contact_keep(const contact_args& a, int64_t n, double y_lo, double y_hi,
                               uint32_t* keep, hipStream_t st) {
  if (n == 0) return hipSuccess;
  if (n < 0 || n > a.capacity) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_contact_keep, grid_for(n), dim3(256), 0, st, a, n, y_lo, y_hi, keep);
  return hipGetLastError();
}

hipError_t launch_contact_compact(int64_t capacity, const contact_slots& src,
                                  const contact_slots& dst, const uint32_t* keep,
                                  const int64_t* off, hipStream_t st) {
  if (capacity == 0) return hipSuccess;
  hipLaunchKernelGGL(k_contact_compact, grid_for(capacity), dim3(256), 0, st, capacity, src, dst,
                     keep, off);
  return hipGetLastError();
}

hipError_t launch_contact_move(const contact_args& a, const contact_move_args& m, int64_t n,
                               hipStream_t st) {
  if (n < 0 || n > a.capacity || (m.count[0] > 0 && m.list_n[0] < 1) ||
      (m.count[1] > 0 && m.list_n[1] < 1))
    return hipErrorInvalidValue;
  const int64_t n_tiles = (n + SCAN_TILE - 1) / SCAN_TILE;
  const int64_t fresh = (m.count[0] + m.count[1] + SCAN_THREADS - 1) / SCAN_THREADS;
  if (n_tiles > 0)
    hipLaunchKernelGGL(k_contact_count, dim3((unsigned)n_tiles), dim3(SCAN_THREADS), 0, st, m);
  hipLaunchKernelGGL(k_contact_offsets, dim3(1), dim3(SCAN_THREADS), 0, st, m, n_tiles);
  if (n_tiles + fresh > 0)
    hipLaunchKernelGGL(k_contact_move, dim3((unsigned)(n_tiles + fresh)), dim3(SCAN_THREADS), 0, st, a,
                       m, n_tiles);
  return hipGetLastError();
}

hipError_t launch_contact_inject(const contact_args& a, const int64_t* base, int64_t count,
                                 const int32_t* sites, int64_t n_sites, uint64_t* next_id,
                                 double t_now, int64_t* n_live, hipStream_t st) {
  if (count > 0) {
    if (n_sites < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_contact_inject, grid_for(count), dim3(256), 0, st, a, base, count, sites,
                       n_sites, (const uint64_t*)next_id, t_now);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_contact_finish, dim3(1), dim3(64), 0, st, base, count, a.capacity, next_id,
                     n_live);
  return hipGetLastError();
}

}  // namespace cntkmc
