// observables.hip -- cell list, overlap tests, pair histograms and Widom
// insertions on one replica's configuration.
//
// Every neighbour search runs on an "observable grid": an unshifted cell grid
// whose side is at least the cutoff of the question asked (1 for overlaps and
// Widom, 1/sf for a compression by sf, rmax for the histograms), stored in
// CSR form (cell start offsets, particle ids and FP64 positions sorted by
// cell).  Because the side covers the cutoff, the set of pairs examined is
// every pair within the cutoff, which is also the set the reference examines
// through its own cell list whenever its cells are at least that wide
// (compute_press.c:61-69 enforces it for the contact histogram).
#include <math.h>

#include <algorithm>
#include <vector>

#include "ctx.h"
#include "device_common.h"

using namespace hsmc;

namespace {

enum Slot { S_CNT = 0, S_START, S_CELLOF, S_IDS, S_PX, S_PY, S_PZ, S_Q0, S_Q1, S_Q2, S_OUT0,
            S_PART, S_BINS, S_SUMS };

struct Grid {
  int nx, ny, nz;
  double sx, sy, sz;
  double ix, iy, iz;  // 1.0 / sx ...
  double lx, ly, lz;
  const int *start;   // C + 1
  const int *ids;     // N, particle id by sorted position
  const double *px, *py, *pz;
  __device__ __forceinline__ int begin(int c) const { return start[c]; }
  __device__ __forceinline__ int end(int c) const { return start[c + 1]; }
};

// EXACT: the reference's cells (cell_part_idx, for cell_list) and sx its cell
// side; otherwise a search grid and sx the reciprocal of its side.
template <bool EXACT>
__global__ void k_grid_count(const double *__restrict__ x, const double *__restrict__ y,
                             const double *__restrict__ z, int n, int nx, int ny, int nz, double sx,
                             double sy, double sz, int *__restrict__ cnt, int2 *__restrict__ cellof) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  auto cell = [](double p, double s, int g) { return EXACT ? plain_cell(p, s, g) : search_cell(p, s, g); };
  const int c = (cell(x[i], sx, nx) * ny + cell(y[i], sy, ny)) * nz + cell(z[i], sz, nz);
  cellof[i] = make_int2(c, atomicAdd(&cnt[c], 1));  // its cell and its place there
}

// Exclusive prefix sum of cnt[0..n) into start[0..n], one workgroup.  Each
// pass covers 32 * 1024 entries: a thread loads its 32 consecutive entries
// at once (all loads in flight together), the waves scan the thread sums in
// registers and the 16 wave totals go through LDS; a carry links the passes.
// CLEAR: the counts are set to zero once read, for the next grid.
template <bool CLEAR>
__global__ void __launch_bounds__(1024) k_scan1(int *__restrict__ cnt, int n, int *__restrict__ start) {
  constexpr int K = 32;
  __shared__ int tot[2][16];
  const int t = threadIdx.x, w = t >> 6;
  int carry = 0;
  for (int base = 0, pass = 0; base < n; base += K * 1024, ++pass) {
    // short scans spread over all threads: k entries each, at most K
    const int k1 = min(K, (n - base + 1023) / 1024);
    const int b = base + t * k1;
    int v[K];
    int s = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      v[k] = (k < k1 && b + k < n) ? cnt[b + k] : 0;
      s += v[k];
    }
    const int incl = group_inclusive_sum<64>(s);
    if ((t & 63) == 63) tot[pass & 1][w] = incl;
    __syncthreads();  // one barrier a pass: the next pass writes the other row
    int before = 0, total = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int u = tot[pass & 1][i];
      before += i < w ? u : 0;
      total += u;
    }
    int run = carry + before + incl - s;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (k < k1 && b + k < n) {
        start[b + k] = run;
        if (CLEAR) cnt[b + k] = 0;
      }
      run += v[k];
    }
    carry += total;
  }
  if (t == 0) start[n] = carry;
}

// Exclusive prefix sum over many workgroups: each 256-thread workgroup scans
// a tile of 4096 entries (16 consecutive per thread) and writes the tile
// total; the totals are scanned by k_scan1; k_scan_add adds each tile's
// offset.  Three short launches in place of one workgroup walking the whole
// array.
constexpr int kScanTile = 4096;
// Up to here k_scan1 alone: 3 us for up to 2000 entries, 5 for 5500, 8 for
// 11700, 16 for 16000 and 25 for 31000, against 9 to 11 for the three launches.
constexpr int kScanOne = 12 * 1024;

template <bool CLEAR>
__global__ void __launch_bounds__(256) k_scan_tile(int *__restrict__ in, int n,
                                                   int *__restrict__ out, int *__restrict__ part) {
  __shared__ int wsum[4];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const long base = (long)blockIdx.x * kScanTile + (long)t * 16;
  int v[16];
  int s = 0;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    v[k] = (base + k < n) ? in[base + k] : 0;
    s += v[k];
  }
  int incl = s;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(incl, d, 64);
    if (lane >= d) incl += u;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  int woff = 0;
  for (int i = 0; i < w; ++i) woff += wsum[i];
  int run = woff + incl - s;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    if (base + k < n) {
      out[base + k] = run;
      if (CLEAR) in[base + k] = 0;
    }
    run += v[k];
  }
  if (t == 255) part[blockIdx.x] = woff + incl;
}

__global__ void k_scan_empty(int *__restrict__ out) {
  if (threadIdx.x == 0) out[0] = 0;
}

__global__ void __launch_bounds__(256) k_scan_add(int *__restrict__ out, int n,
                                                  const int *__restrict__ offs, int tiles) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] += offs[i / kScanTile];
  if (i == 0) out[n] = offs[tiles];
}

__global__ void k_grid_scatter(const double *__restrict__ x, const double *__restrict__ y,
                               const double *__restrict__ z, int n, const int2 *__restrict__ cellof,
                               const int *__restrict__ start, int *__restrict__ ids, double *__restrict__ px,
                               double *__restrict__ py, double *__restrict__ pz) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int2 c = cellof[i];
  const int pos = start[c.x] + c.y;
  if (ids) ids[pos] = i;
  px[pos] = x[i];
  py[pos] = y[i];
  pz[pos] = z[i];
}

// One thread per cell: ascending ids, then the reference's part_cell row
// [count, ids..., -1...] (cell_list.c:148-171).
__global__ void k_part_cell(const int *__restrict__ start, int C, int *__restrict__ ids,
                            int max_part, int *__restrict__ out, unsigned *__restrict__ err) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int b = start[c], n = start[c + 1] - start[c];
  int *row = out + (size_t)c * max_part;
  if (n > max_part - 1) {  // cell_list_check (cell_list.c:229-232)
    atomicOr(err, kErrOverflow);
    row[0] = n;
    return;
  }
  for (int i = 1; i < n; ++i) {  // insertion sort of a few ids
    const int v = ids[b + i];
    int j = i - 1;
    while (j >= 0 && ids[b + j] > v) {
      ids[b + j + 1] = ids[b + j];
      --j;
    }
    ids[b + j + 1] = v;
  }
  row[0] = n;
  for (int j = 1; j < max_part; ++j) row[j] = (j <= n) ? ids[b + j - 1] : -1;
}

// Iterate the distinct cells of the 27-stencil around (cx,cy,cz).
template <class F>
__device__ __forceinline__ bool for_stencil(const Grid &g, int cx, int cy, int cz, F &&f) {
  for (int dx = -1; dx <= 1; ++dx) {
    if (!stencil_axis_ok(dx, g.nx)) continue;
    const int ax = wrap_index(cx + dx, g.nx);
    for (int dy = -1; dy <= 1; ++dy) {
      if (!stencil_axis_ok(dy, g.ny)) continue;
      const int ay = wrap_index(cy + dy, g.ny);
      for (int dz = -1; dz <= 1; ++dz) {
        if (!stencil_axis_ok(dz, g.nz)) continue;
        const int c = (ax * g.ny + ay) * g.nz + wrap_index(cz + dz, g.nz);
        if (f(g.start[c], g.start[c + 1])) return true;
      }
    }
  }
  return false;
}

// Any sphere other than skip_id closer than 1 to q, in the 27 cells around
// q (check_overlap, moves.c:157-212, and widom_check_overlap,
// compute_widom_chem_pot.c:82-120).  The answer does not depend on the
// order of the cells, so they are visited nearest first (the point's own
// cell, then the 6 sharing a face, then the rest), with the ranges of the
// first 7 loaded together: a point that overlaps usually does so there, and
// leaves after one round trip for the ranges and one for the spheres.
template <bool SKIP, class G>
__device__ __forceinline__ bool point_overlaps(const G &g, double qx, double qy, double qz,
                                               int skip_id) {
  const int cx = search_cell(qx, g.ix, g.nx), cy = search_cell(qy, g.iy, g.ny),
            cz = search_cell(qz, g.iz, g.nz);
  auto cell_of = [&](int j, bool &ok) {
    int dx, dy, dz;
    stencil_by_distance(j, dx, dy, dz);
    ok = stencil_axis_ok(dx, g.nx) && stencil_axis_ok(dy, g.ny) && stencil_axis_ok(dz, g.nz);
    return ok ? (wrap_index(cx + dx, g.nx) * g.ny + wrap_index(cy + dy, g.ny)) * g.nz +
                    wrap_index(cz + dz, g.nz)
              : 0;
  };
  auto scan = [&](int b, int e) {
    for (int p = b; p < e; ++p) {
      // the id and the position load together; the skip is tested after
      int id = 0;
      if constexpr (SKIP) id = g.ids[p];
      const double d2 = dist2(qx, qy, qz, g.px[p], g.py[p], g.pz[p], g.lx, g.ly, g.lz);
      if ((!SKIP || id != skip_id) && d2 < 1.0) return true;
    }
    return false;
  };
  int c7[7], b7[7], e7[7];
  bool ok7[7];
#pragma unroll
  for (int j = 0; j < 7; ++j) c7[j] = cell_of(j, ok7[j]);
#pragma unroll
  for (int j = 0; j < 7; ++j) b7[j] = g.begin(c7[j]);
#pragma unroll
  for (int j = 0; j < 7; ++j) e7[j] = g.end(c7[j]);
#pragma unroll
  for (int j = 0; j < 7; ++j)
    if (!ok7[j]) e7[j] = b7[j];  // a cell the stencil leaves out (tiny grids): empty
#pragma unroll
  for (int j = 0; j < 7; ++j)
    if (scan(b7[j], e7[j])) return true;
  for (int j = 7; j < 27; ++j) {
    bool ok;
    const int c = cell_of(j, ok);
    if (ok && scan(g.begin(c), g.end(c))) return true;
  }
  return false;
}

__global__ void k_overlap_batch(Grid g, const int *__restrict__ idx, const double *__restrict__ q,
                                int m, unsigned char *__restrict__ out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= m) return;
  out[k] = point_overlaps<true>(g, q[3 * k], q[3 * k + 1], q[3 * k + 2], idx[k]) ? 1 : 0;
}

// A few queries without a grid: a workgroup per query tests its sphere against
// all N, the same tests in another order.  The queries come by value, the
// answers go to pinned memory: one launch and one wait, where a grid of a
// configuration not seen before costs three launches and the queries two
// copies.  A call after a move of one sphere, by grid and so: 82 and 24 us at N
// = 256 (18 of them the query), 82 and 28 at 16384; on a grid that is there 44
// and 18, 44 and 23.  (Workgroups of 256 take as long up to N = 256.)
constexpr int kFewQueries = 8;
constexpr int kFewSpheres = 16384;

struct FewQueries {
  double q[kFewQueries][3];
  int idx[kFewQueries];
};

__global__ void __launch_bounds__(1024)
k_overlap_few(FewQueries f, const double *__restrict__ x, const double *__restrict__ y,
              const double *__restrict__ z, int n, double lx, double ly, double lz,
              unsigned long long *__restrict__ host) {
  const int k = blockIdx.x;
  const double qx = f.q[k][0], qy = f.q[k][1], qz = f.q[k][2];
  const int skip = f.idx[k];
  int hit = 0;
#pragma unroll 4
  for (int i = threadIdx.x; i < n; i += (int)blockDim.x)
    hit |= (dist2(qx, qy, qz, x[i], y[i], z[i], lx, ly, lz) < 1.0) & (i != skip);
  hit = __syncthreads_or(hit);
  if (threadIdx.x == 0) host[k] = hit ? 1ull : 0ull;
}

__global__ void k_widom_points(Grid g, const double *__restrict__ q, int m,
                               unsigned char *__restrict__ out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= m) return;
  out[k] = point_overlaps<false>(g, q[3 * k], q[3 * k + 1], q[3 * k + 2], -1) ? 0 : 1;
}

// ---- results of a launch ----------------------------------------------------
// Each workgroup stores its counts in its own row of `part` and one more
// kernel adds the rows up into the context's pinned host memory, so a call is
// its kernels and one wait: nothing to clear, no copy.  (An atomic on one
// address from workgroups on different XCDs takes about 0.1 us, one after
// the other: 512 workgroups adding to shared counts took 70 us longer.)

// Column sums of rows x cols counts: 64 columns a workgroup, 16 interleaved
// groups of rows; with several workgroups along y each takes its share of
// the rows and stores its own row of sums.
template <class T>
__global__ void __launch_bounds__(1024)
k_sum_rows(const T *__restrict__ part, int rows, int cols, unsigned long long *__restrict__ out) {
  __shared__ unsigned long long s[16][64];
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6, c = blockIdx.x * 64 + lane;
  const int cc = min(c, cols - 1);
  unsigned long long v = 0;
#pragma unroll 8
  for (int r = blockIdx.y * 16 + q; r < rows; r += 16 * gridDim.y) v += part[(size_t)r * cols + cc];
  s[q][lane] = v;
  __syncthreads();
  if (q) return;
#pragma unroll
  for (int k = 1; k < 16; ++k) v += s[k][lane];
  if (c < cols) out[(size_t)blockIdx.y * cols + c] = v;
}

// Sum (or OR) of n 64-bit values; with err, the sticky error bits too.
template <bool OR>
__global__ void __launch_bounds__(1024)
k_sum_all(const unsigned long long *__restrict__ part, int n, const unsigned *__restrict__ err,
          unsigned long long *__restrict__ host) {
  __shared__ unsigned long long s[16];
  unsigned long long v = 0;
#pragma unroll 8
  for (int i = threadIdx.x; i < n; i += 1024) v = OR ? v | part[i] : v + part[i];
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long u = __shfl_xor(v, o, 64);
    v = OR ? v | u : v + u;
  }
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x) return;
  for (int k = 1; k < 16; ++k) v = OR ? v | s[k] : v + s[k];
  host[0] = v;
  if (err) host[1] = *err;
}

__device__ __forceinline__ unsigned long long block_sum_u64(unsigned long long v) {
  __shared__ unsigned long long red[16];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (l == 0) red[w] = v;
  __syncthreads();
  unsigned long long s = 0;
  if (threadIdx.x == 0) {
    for (int i = 0; i < (int)((blockDim.x + 63) >> 6); ++i) s += red[i];
  }
  return s;
}

// widom_insertion (compute_widom_chem_pot.c:44-71) on a Philox stream:
// point i has counter {i_lo, i_hi, sample_lo, 0x5749xxxx}, coordinates
// u/(2^32-1) * L (widom_rand_pos, :73-80).
constexpr int kWidomUniformBlocks = 8192;

template <class G>
__device__ __forceinline__ void uniform_points(const G &g, uint32_t k0, uint32_t k1,
                                               unsigned long long sample, long long first,
                                               long long n, unsigned long long *__restrict__ part) {
  unsigned long long h = 0;
  const long long stride = (long long)gridDim.x * blockDim.x;
  const uint32_t c3 = 0x57490000u | (uint32_t)((sample >> 32) & 0xFFFFu);
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += stride) {
    const unsigned long long i = (unsigned long long)(first + t);
    uint32_t u[4];
    philox4x32_10((uint32_t)i, (uint32_t)(i >> 32), (uint32_t)sample, c3, k0, k1, u);
    const double qx = u32_unit_closed(u[0]) * g.lx;
    const double qy = u32_unit_closed(u[1]) * g.ly;
    const double qz = u32_unit_closed(u[2]) * g.lz;
    if (!point_overlaps<false>(g, qx, qy, qz, -1)) ++h;
  }
  const unsigned long long s = block_sum_u64(h);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ void __launch_bounds__(256)
k_widom_uniform(Grid g, uint32_t k0, uint32_t k1, unsigned long long sample, long long first,
                long long n, unsigned long long *__restrict__ part) {
  uniform_points(g, k0, k1, sample, first, n, part);
}

// The same for systems whose grid and positions fit in LDS: every workgroup
// files the spheres itself (a few us, beside the three launches of
// a grid in memory) and its points' scattered reads stay on the chip.
constexpr int kWidomLdsThreads = 512, kWidomLdsBlocks = 1024;

struct LdsGrid {  // after filing, last[c] is the end of cell c and so the start of cell c + 1
  int nx, ny, nz;
  double ix, iy, iz, lx, ly, lz;
  const int *last;
  const double *px, *py, *pz;
  __device__ __forceinline__ int begin(int c) const { return c ? last[c - 1] : 0; }
  __device__ __forceinline__ int end(int c) const { return last[c]; }
};

size_t widom_lds_bytes(long N, long C) { return sizeof(double) * 3 * N + sizeof(int) * C; }

template <int THREADS>
__global__ void __launch_bounds__(THREADS)
k_widom_uniform_lds(Grid gg, int N, const double *__restrict__ x, const double *__restrict__ y,
                    const double *__restrict__ z, uint32_t k0, uint32_t k1,
                    unsigned long long sample, long long first, long long n,
                    unsigned long long *__restrict__ part) {
  extern __shared__ double lds_pos[];
  __shared__ int tot[THREADS / 64];
  double *px = lds_pos, *py = px + N, *pz = py + N;
  int *cnt = reinterpret_cast<int *>(pz + N);
  const int t = threadIdx.x, C = gg.nx * gg.ny * gg.nz;
  for (int c = t; c < C; c += THREADS) cnt[c] = 0;
  __syncthreads();
  auto cell = [&](double a, double b, double c) {
    return (search_cell(a, gg.ix, gg.nx) * gg.ny + search_cell(b, gg.iy, gg.ny)) * gg.nz +
           search_cell(c, gg.iz, gg.nz);
  };
  for (int i = t; i < N; i += THREADS) atomicAdd(&cnt[cell(x[i], y[i], z[i])], 1);
  __syncthreads();
  // counts to starts: a run of consecutive cells per thread
  const int per = (C + THREADS - 1) / THREADS, c0 = min(t * per, C), c1 = min(c0 + per, C);
  int s = 0;
  for (int c = c0; c < c1; ++c) s += cnt[c];
  const int incl = group_inclusive_sum<64>(s);
  if ((t & 63) == 63) tot[t >> 6] = incl;
  __syncthreads();
  int run = incl - s;
  for (int w = 0; w < (t >> 6); ++w) run += tot[w];
  for (int c = c0; c < c1; ++c) {
    const int k = cnt[c];
    cnt[c] = run;
    run += k;
  }
  __syncthreads();
  for (int i = t; i < N; i += THREADS) {
    const double a = x[i], b = y[i], c = z[i];
    const int p = atomicAdd(&cnt[cell(a, b, c)], 1);
    px[p] = a;
    py[p] = b;
    pz[p] = c;
  }
  __syncthreads();
  const LdsGrid g{gg.nx, gg.ny, gg.nz, gg.ix, gg.iy, gg.iz, gg.lx, gg.ly, gg.lz, cnt, px, py, pz};
  uniform_points(g, k0, k1, sample, first, n, part);
}

// Cell-stratified uniform insertion: every cell of the observable grid
// (side >= 1) receives `per_cell` points uniform inside it.  The cells have
// equal volume, so hits / (per_cell * C) is an unbiased estimate of the
// insertion probability, like widom_insertion's uniform points
// (compute_widom_chem_pot.c:44-80), with a variance no larger.  Point j of
// cell c comes from Philox counter {c, j, sample_lo, 0x5743xxxx}:
// coordinate (ic + (u + 0.5) 2^-32) * side per axis.
//
// One wave per cell: lanes j < 27 read the neighbour cells' ranges, and the
// spheres of the 27 cells are staged once in LDS in the order own cell, 6
// faces, 12 edges, 8 corners (the likeliest overlaps first).  The wave then
// takes 128 points at a time, two to a lane, and walks the list in lockstep
// (every lane reads entry e together: an LDS broadcast), leaving the walk as
// soon as a ballot shows every point overlapping.
//
// Bounded by instructions: per cell the points' draws (20 32 x 32-bit
// products each) and 26 tests of up to 128 points.  The list therefore holds
// positions relative to the cell, image applied, in FP32: a test is 6.5
// instructions and one 16-byte read, where the FP64 one is 9 (or 15 with the
// minimum image) and three reads.  A smallest squared distance within
// kWidomBand of 1 is decided again by the reference's FP64 arithmetic
// (moves.c:400-431 order, minimum image) on the FP64 positions, so every
// decision is the FP64 one: cells are less than 2 wide (floor(L) of them), so
// a sphere less than 2 away lies within 4 of the cell's corner, each
// coordinate within 3e-7 of its value, a difference within 7e-7 and the
// squared distance within 3e-6 of its own near 1.  Axes of fewer than 3 cells,
// where a neighbour cell's image depends on the point, take the FP64 test.
// A call of 10^7 insertions at N = 108000 on a grid that is there: 82 us, 100
// with FP64 tests, 139 with 64-bit cell arithmetic and a wave's set-up for
// every cell besides (6144 workgroups take several cells a wave; 2048 of them
// 84 us, a wave for each cell 103); 1000 a cell at N = 4000 39, 68 and 67.
constexpr int kWidomCellsLcap = 256;   // bound of spheres in a 27-cell stencil (host-checked)
constexpr int kWidomCellsWaves = 4;    // waves per workgroup
constexpr int kWidomCellsBlocks = 6144;
constexpr float kWidomBand = 1e-5f;

template <bool FAST>
__global__ void __launch_bounds__(64 * kWidomCellsWaves)
k_widom_cells(Grid g, uint32_t k0, uint32_t k1, unsigned long long sample, int per_cell,
              unsigned long long *__restrict__ part, unsigned *__restrict__ err) {
  __shared__ float4 list[FAST ? kWidomCellsWaves : 1][FAST ? kWidomCellsLcap : 1];
  __shared__ double exact[FAST ? 1 : kWidomCellsWaves][3][FAST ? 1 : kWidomCellsLcap];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int C = g.nx * g.ny * g.nz;  // at most 2^28 (build_grid)
  int dx = 0, dy = 0, dz = 0;        // lane < 27: its neighbour cell (distinct cells only)
  if (lane < 27) stencil_by_distance(lane, dx, dy, dz);
  const bool near = lane < 27 && stencil_axis_ok(dx, g.nx) && stencil_axis_ok(dy, g.ny) && stencil_axis_ok(dz, g.nz);
  const uint32_t c3 = 0x57430000u | (uint32_t)((sample >> 32) & 0xFFFFu);
  const float sfx = (float)(g.sx * 0x1p-32), sfy = (float)(g.sy * 0x1p-32), sfz = (float)(g.sz * 0x1p-32);
  unsigned long long h = 0;
  for (int c = blockIdx.x * kWidomCellsWaves + w; c < C; c += gridDim.x * kWidomCellsWaves) {
    const int t2 = c / g.nz, iz = c - t2 * g.nz, ix = t2 / g.ny, iy = t2 - ix * g.ny;
    int b = 0, n = 0;
    if (near) {
      const int jx = ix + dx, jy = iy + dy, jz = iz + dz;
      const int nc = (wrap_index(jx, g.nx) * g.ny + wrap_index(jy, g.ny)) * g.nz + wrap_index(jz, g.nz);
      b = g.start[nc];
      n = g.start[nc + 1] - b;
    }
    const int incl = group_inclusive_sum<32>(n);
    // the list length, read into a scalar register so that the point loop
    // below is a uniform loop; padded to a multiple of 4 with positions no
    // point can overlap (the loop tests 4 entries between its exit checks)
    const int T = __builtin_amdgcn_readlane(incl, 26);
    const int T4 = (T + 3) & ~3;
    if (T4 > kWidomCellsLcap) {  // above the packing bound the host checks: cannot happen
      if (lane == 0) atomicOr(err, kErrListFull);
      continue;
    }
    const int o = incl - n;
    if constexpr (FAST) {
      // the entries' places first, by cells; then an entry to a lane, so that
      // three loads fetch the list and not three for each sphere of a cell
#pragma unroll 1
      for (int q = 0; q < n; ++q) list[w][o + q].w = __int_as_float(b + q);
      wave_lds_sync();
      const double cx = (ix + 0.5) * g.sx, cy = (iy + 0.5) * g.sy, cz = (iz + 0.5) * g.sz;
      auto from_corner = [](double v, double centre, double side, double L) {
        const double d = v - centre;
        return (float)(d - (__builtin_fabs(d) > 0.5 * L ? __builtin_copysign(L, d) : 0.0) + 0.5 * side);
      };
#pragma unroll 1
      for (int e = lane; e < T4; e += 64) {
        const int s = e < T ? __float_as_int(list[w][e].w) : 0;
        const double px = g.px[s], py = g.py[s], pz = g.pz[s];
        list[w][e].x = e < T ? from_corner(px, cx, g.sx, g.lx) : 1e18f;
        list[w][e].y = from_corner(py, cy, g.sy, g.ly);
        list[w][e].z = from_corner(pz, cz, g.sz, g.lz);
      }
    } else {
      for (int q = 0; q < n; ++q) {
        exact[w][0][o + q] = g.px[b + q];
        exact[w][1][o + q] = g.py[b + q];
        exact[w][2][o + q] = g.pz[b + q];
      }
      if (lane < T4 - T) exact[w][0][T + lane] = exact[w][1][T + lane] = exact[w][2][T + lane] = 1e300;
    }
    wave_lds_sync();
    // point jj of the cell
    auto draw = [&](int jj, uint32_t u[4]) {
      philox4x32_10((uint32_t)c, (uint32_t)jj, (uint32_t)sample, c3, k0, k1, u);
    };
    auto coord = [](int i, uint32_t u, double side) { return ((double)i + ((double)u + 0.5) * 0x1p-32) * side; };
    auto walk = [&](auto points, int base) {
      constexpr int P = decltype(points)::value;
      bool mine[P];
      if constexpr (FAST) {
        float q[P][3], m[P];
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const int jj = base + 64 * p + lane;
          uint32_t u[4];
          draw(jj, u);
          q[p][0] = (float)u[0] * sfx;
          q[p][1] = (float)u[1] * sfy;
          q[p][2] = (float)u[2] * sfz;
          mine[p] = jj < per_cell;
          m[p] = mine[p] ? 9.0f : 0.0f;
        }
        for (int e = 0; e < T4; e += 4) {
#pragma unroll
          for (int i = 0; i < 4; i += 2) {
            const float4 a = list[w][e + i], d = list[w][e + i + 1];
#pragma unroll
            for (int p = 0; p < P; ++p) {
              const float ax = q[p][0] - a.x, ay = q[p][1] - a.y, az = q[p][2] - a.z;
              const float bx = q[p][0] - d.x, by = q[p][1] - d.y, bz = q[p][2] - d.z;
              m[p] = fminf(m[p], fminf(__builtin_fmaf(az, az, __builtin_fmaf(ay, ay, ax * ax)),
                                       __builtin_fmaf(bz, bz, __builtin_fmaf(by, by, bx * bx))));
            }
          }
          float far = m[0];
          if constexpr (P == 2) far = fmaxf(m[0], m[1]);
          if (__all(far < 1.0f - kWidomBand)) break;
        }
#pragma unroll
        for (int p = 0; p < P; ++p) {
          bool free = m[p] >= 1.0f + kWidomBand;
          const bool undecided = m[p] >= 1.0f - kWidomBand && !free;
          if (__any(undecided)) {
            uint32_t u[4];
            draw(base + 64 * p + lane, u);
            const double x = coord(ix, u[0], g.sx), y = coord(iy, u[1], g.sy), z = coord(iz, u[2], g.sz);
            if (undecided)
              free = true;
#pragma unroll 1
            for (int e = 0; e < T; ++e) {
              const int s = __float_as_int(list[w][e].w);
              if (undecided && dist2(x, y, z, g.px[s], g.py[s], g.pz[s], g.lx, g.ly, g.lz) < 1.0) free = false;
            }
          }
          if (free && mine[p]) ++h;
        }
      } else {
        double q[P][3], m[P];
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const int jj = base + 64 * p + lane;
          uint32_t u[4];
          draw(jj, u);
          q[p][0] = coord(ix, u[0], g.sx);
          q[p][1] = coord(iy, u[1], g.sy);
          q[p][2] = coord(iz, u[2], g.sz);
          mine[p] = jj < per_cell;
          m[p] = mine[p] ? 1e300 : 0.0;
        }
        for (int e = 0; e < T4; ++e) {
#pragma unroll
          for (int p = 0; p < P; ++p)
            m[p] = fmin(m[p], dist2(q[p][0], q[p][1], q[p][2], exact[w][0][e], exact[w][1][e], exact[w][2][e], g.lx,
                                    g.ly, g.lz));
        }
#pragma unroll
        for (int p = 0; p < P; ++p)
          if (m[p] >= 1.0) ++h;
      }
    };
    int base = 0;
    if constexpr (FAST)
      for (; base + 64 < per_cell; base += 128) walk(std::integral_constant<int, 2>{}, base);
    for (; base < per_cell; base += 64) walk(std::integral_constant<int, 1>{}, base);
    __builtin_amdgcn_wave_barrier();  // the list is rewritten for the next cell
  }
  const unsigned long long s = block_sum_u64(h);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// check_overlap(idx, sf, sf, sf) (moves.c:157-212) for each query.
__global__ void k_overlap_scaled(Grid g, const double *__restrict__ x, const double *__restrict__ y,
                                 const double *__restrict__ z, const int *__restrict__ idx,
                                 const double *__restrict__ sfv, int m,
                                 unsigned char *__restrict__ out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= m) return;
  const int i = idx[k];
  const double sf = sfv[k];
  const double ax = x[i], ay = y[i], az = z[i];
  const int cx = search_cell(ax, g.ix, g.nx), cy = search_cell(ay, g.iy, g.ny), cz = search_cell(az, g.iz, g.nz);
  const bool ov = for_stencil(g, cx, cy, cz, [&](int b, int e) {
    for (int p = b; p < e; ++p) {
      if (g.ids[p] == i) continue;
      if (dist2_scaled(ax, ay, az, g.px[p], g.py[p], g.pz[p], g.lx, g.ly, g.lz, sf) < 1.0)
        return true;
    }
    return false;
  });
  out[k] = ov ? 1 : 0;
}

__global__ void k_pair_dist(const double *__restrict__ x, const double *__restrict__ y,
                            const double *__restrict__ z, const int *__restrict__ ii,
                            const int *__restrict__ jj, int m, double sf, double lx, double ly,
                            double lz, double *__restrict__ out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= m) return;
  const int i = ii[k], j = jj[k];
  out[k] = sqrt(dist2_scaled(x[i], y[i], z[i], x[j], y[j], z[j], lx, ly, lz, sf));
}

// ---- pair kernels --------------------------------------------------------
// What a histogram kernel asks of a pair: dr < rmax_eff and bin
// (int)((dr - 1.0) / dr_bin) (compute_rdf.c:118-124, compute_press.c:150-155).
// dr, the difference and the quotient are correctly rounded and so grow with
// the squared distance s: dr < rmax_eff is s < smax, and the bin is b when
// edge[b] <= s < edge[b + 1], with smax and the edges the first doubles past
// each step, which the host finds with the formula itself.  A pair is binned
// by an FP32 estimate corrected against the edges, about 15 instructions in
// place of the 50 of an FP64 square root and division.
struct Bins {
  double dr_bin, rmax_eff, smax;
  float inv_bin;
  int n;
  const double *edge;  // n + 1 entries, or null: few bins, binned by the formula
};

// The kernels' LDS: nbins counts, then the edges.
__device__ __forceinline__ double *hist_edges(unsigned int *hist, int n) {
  return reinterpret_cast<double *>(hist + ((n + 1) & ~1));
}

__device__ __forceinline__ void hist_begin(const Bins &bn, unsigned int *hist) {
  for (int b = threadIdx.x; b < bn.n; b += blockDim.x) hist[b] = 0;
  if (bn.edge) {
    double *e = hist_edges(hist, bn.n);
    for (int b = threadIdx.x; b <= bn.n; b += blockDim.x) e[b] = bn.edge[b];
  }
  __syncthreads();
}

template <bool EDGES>
__device__ __forceinline__ void bin_pair(const Bins &bn, unsigned int *hist, double s,
                                         unsigned long long &bad) {
  if (!(s < bn.smax)) return;
  int b;
  bool in;
  if constexpr (EDGES) {
    const double *e = hist_edges(hist, bn.n);
    b = (int)((__builtin_amdgcn_sqrtf((float)s) - 1.0f) * bn.inv_bin);
    b = min(max(b, 0), bn.n - 1);
    const double lo = e[b], hi = e[b + 1];
    in = s >= lo && s < hi;
    if (!in) {  // next to an edge, or out of the bins' range
      while (b > 0 && s < e[b]) --b;
      while (b < bn.n - 1 && s >= e[b + 1]) ++b;
      in = s >= e[b] && s < e[b + 1];
    }
  } else {
    b = (int)((sqrt(s) - 1.0) / bn.dr_bin);
    in = b >= 0 && b < bn.n;
  }
  if (in)
    atomicAdd(&hist[b], 1u);
  else
    ++bad;
}

// The workgroup's counts, and its pairs out of the bins' range, in its row:
// these in two words, as one workgroup can meet more than 2^32 of them (a cell
// of a cutoff of 0.4 box edges at N = 2 * 10^6).
__device__ __forceinline__ void hist_end(const Bins &bn, const unsigned int *hist, unsigned long long bad,
                                         unsigned int *__restrict__ part) {
  unsigned int *row = part + (size_t)blockIdx.x * (bn.n + 2);
  const unsigned long long out = block_sum_u64(bad);  // with the barrier before the counts are read
  for (int b = threadIdx.x; b < bn.n; b += blockDim.x) row[b] = hist[b];
  if (threadIdx.x == 0) {
    row[bn.n] = (unsigned int)out;
    row[bn.n + 1] = (unsigned int)(out >> 32);
  }
}

// Scale factors of one scan, passed by value (no host-to-device copy).
struct SfTable {
  double v[64];
};

// Bits k of the factors at which a pair overlaps after scaling.  s0 is its
// unscaled squared distance: at cut2 and beyond no factor makes it overlap.
__device__ __forceinline__ void scaled_pair(const SfTable &sf, int nsf, double cut2, double s0,
                                            double ax, double ay, double az, double bx, double by,
                                            double bz, double lx, double ly, double lz,
                                            unsigned long long &m) {
  if (s0 >= cut2) return;
  for (int k = 0; k < nsf; ++k)
    if (dist2_scaled(ax, ay, az, bx, by, bz, lx, ly, lz, sf.v[k]) < 1.0) m |= 1ull << k;
}

__device__ __forceinline__ void mask_end(unsigned long long m, unsigned long long *__restrict__ part) {
  __shared__ unsigned long long red[16];
  for (int o = 32; o > 0; o >>= 1) m |= __shfl_xor(m, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x) return;
  for (int k = 1; k < (int)(blockDim.x >> 6); ++k) m |= red[k];
  part[blockIdx.x] = m;
}

// All pairs of N spheres without a grid, for systems of up to kAllPairs
// spheres (kAllPairsWide for a cutoff of kWide and more): a wave takes 64 spheres, one a lane, against a run of JC spheres
// read through the scalar cache (their index is the same in every lane), and
// keeps the pairs of a later sphere.  f(squared distance, ...) of each pair.
// A grid costs three launches and a stencil walk of dependent loads; all
// 8 M pairs of 4000 spheres are 15 FP64 instructions each on the whole GPU:
// contact histogram 11.5 us (27.0 with a thread per sphere on a grid, and the
// grid 26), g(r) to 5 diameters 14.5 us (130 with a wave per pair of cells),
// 20 scale factors 12.2 us (28.0).  Whole calls, all pairs against the grid:
// contacts 29.8 / 33.9 us at N = 4000, 34.9 / 34.1 at 5324, 41.8 / 34.9 at
// 6912; g(r) 51.5 / 54.5 us at 6912, about 62 / 62 at 8000.
constexpr int kAllPairs = 5120, kAllPairsWide = 7168;
constexpr double kWide = 4.0;
constexpr int kPairThreads = 512, kPairBlocks = 2048;

template <int JC, class F>
__device__ __forceinline__ void all_pairs(const double *__restrict__ x, const double *__restrict__ y,
                                          const double *__restrict__ z, int n, double lx, double ly,
                                          double lz, F &&f) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (kPairThreads / 64) + (threadIdx.x >> 6)));
  const int waves = gridDim.x * (kPairThreads / 64);
  // tile a of 64 spheres meets tiles a .. nt - 1; tiles a and nt - 1 - a
  // together meet nt + 1, so task t of the half-by-(nt + 1) rectangle is one
  // pair of tiles (the middle tile of an odd number comes up twice: its
  // second half of tasks is left out), JC spheres of the later tile at a time
  const int nt = (n + 63) / 64, tasks = (nt + 1) / 2 * (nt + 1) * (64 / JC);
  for (int t = wave; t < tasks; t += waves) {
    const int u = t / (64 / JC), p = u / (nt + 1), r = u % (nt + 1);
    const bool low = r < nt - p;
    if (!low && nt - 1 - p == p) continue;
    const int a = low ? p : nt - 1 - p, b = low ? p + r : r - 1;
    const int i0 = 64 * a, j0 = 64 * b + (t % (64 / JC)) * JC, j1 = min(j0 + JC, n);
    const int i = i0 + lane;
    const int ic = min(i, n - 1);
    const int after = i < n ? i : n;  // a lane past the end keeps no pair
    const double ax = x[ic], ay = y[ic], az = z[ic];
#pragma unroll 8
    for (int j = j0; j < j1; ++j) {
      const double bx = x[j], by = y[j], bz = z[j];
      const double s = dist2(ax, ay, az, bx, by, bz, lx, ly, lz);
      if (j > after) f(s, ax, ay, az, bx, by, bz);
    }
  }
}

template <int JC, bool EDGES>
__global__ void __launch_bounds__(kPairThreads)
k_hist_all(const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z,
           int n, double lx, double ly, double lz, Bins bn, unsigned int *__restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) unsigned int hist[];
  hist_begin(bn, hist);
  unsigned long long bad = 0;
  all_pairs<JC>(x, y, z, n, lx, ly, lz, [&](double s, double, double, double, double, double, double) {
    bin_pair<EDGES>(bn, hist, s, bad);
  });
  hist_end(bn, hist, bad, part);
}

template <int JC>
__global__ void __launch_bounds__(kPairThreads)
k_scaled_all(const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z,
             int n, double lx, double ly, double lz, SfTable sf, int nsf, double cut2,
             unsigned long long *__restrict__ part) {
  unsigned long long m = 0;
  all_pairs<JC>(x, y, z, n, lx, ly, lz,
                [&](double s, double ax, double ay, double az, double bx, double by, double bz) {
                  scaled_pair(sf, nsf, cut2, s, ax, ay, az, bx, by, bz, lx, ly, lz, m);
                });
  mask_end(m, part);
}

// Pairs of larger systems on a grid whose side is at least cutoff / S and
// which has at least 2 S + 1 cells an axis.  A workgroup takes a cell A: the
// cells of A's stencil that follow it (half of the (2S+1)^3, each pair of
// cells once) are runs along z of consecutive entries of the sorted arrays,
// two where a row wraps.  The runs' spheres go one to a lane, loaded
// contiguously, and the spheres of A, the same for every lane, come through
// the scalar cache.  f(squared distance, ...) of each pair.
// g(r) to 5 diameters at N = 32000 on 12^3 cells: 52 us (244 us with a wave
// per pair of cells 5 wide and each pair binned by square root and division).
// (Four cells a workgroup of 1024 left fewer counts to add up but 75 us of
// uneven work where single cells take 53.)
// At most kRowBlocks workgroups, and so rows of counts: 67 MB with 8192 bins.
constexpr int kRowThreads = 256, kRowBlocks = 2048;

template <int S, class F>
__device__ __forceinline__ void row_pairs(const Grid &g, F &&f) {
  constexpr int ROWS = 2 * S * (S + 1) + 1, RUNS = 2 * ROWS;  // rows after A's, and A's own
  __shared__ int run_b[64], run_off[64];
  const int t = threadIdx.x;
  const int C = g.nx * g.ny * g.nz;
  for (int A = blockIdx.x; A < C; A += gridDim.x) {
    const int bA = g.start[A], eA = g.start[A + 1];
    if (bA == eA) continue;  // the whole workgroup
    const int cx = A / (g.ny * g.nz), cy = (A / g.nz) % g.ny, cz = A % g.nz;
    __syncthreads();  // the previous cell's runs are no longer read
    if (t < 64) {
      int b = 0, len = 0;
      if (t < RUNS) {
        // row 0 is A's own (A and the cells after it along z); row k >= 1
        // the k-th offset (dx, dy) after (0, 0)
        const int k = t >> 1, d = k + S;
        const int dx = d / (2 * S + 1), dy = d % (2 * S + 1) - S;
        const int z0 = k ? cz - S : cz, z1 = cz + S;
        const int base = (wrap_index(cx + dx, g.nx) * g.ny + wrap_index(cy + dy, g.ny)) * g.nz;
        int a0, a1;
        if ((t & 1) == 0) {  // the part inside [0, nz)
          a0 = max(z0, 0), a1 = min(z1, g.nz - 1);
        } else if (z0 < 0) {           // the part that wraps
          a0 = z0 + g.nz, a1 = g.nz - 1;
        } else {
          a0 = 0, a1 = z1 - g.nz;
        }
        if (a1 >= a0) {
          b = g.start[base + a0];
          len = g.start[base + a1 + 1] - b;
        }
      }
      const int incl = group_inclusive_sum<64>(len);
      run_b[t] = b;
      run_off[t] = incl - len;
    }
    __syncthreads();
    const int total = run_off[63];  // runs past RUNS are empty
    // without a wrap every difference is within (S + 1) sides, under half a
    // box of 2 S + 3 cells: the minimum image changes none of them
    const bool direct = g.nx >= 2 * S + 3 && g.ny >= 2 * S + 3 && g.nz >= 2 * S + 3 && cx + S < g.nx &&
                        cy >= S && cy + S < g.ny && cz >= S && cz + S < g.nz;
    for (int j = t; j < total; j += kRowThreads) {
      int r = 0;
#pragma unroll
      for (int w = 32; w > 0; w >>= 1)
        if (run_off[r + w] <= j) r += w;  // the last run that starts at or before j
      const int q = run_b[r] + j - run_off[r];
      const double qx = g.px[q], qy = g.py[q], qz = g.pz[q];
      const int before = q < eA && q >= bA ? q : eA;  // in A itself the spheres before q
      if (direct) {
#pragma unroll 2
        for (int p = bA; p < eA; ++p) {
          const double ax = g.px[p], ay = g.py[p], az = g.pz[p];
          const double dx = ax - qx, dy = ay - qy, dz = az - qz;
          if (p < before) f(dx * dx + dy * dy + dz * dz, ax, ay, az, qx, qy, qz);
        }
      } else {
#pragma unroll 1
        for (int p = bA; p < eA; ++p) {
          const double ax = g.px[p], ay = g.py[p], az = g.pz[p];
          const double s = dist2(ax, ay, az, qx, qy, qz, g.lx, g.ly, g.lz);
          if (p < before) f(s, ax, ay, az, qx, qy, qz);
        }
      }
    }
  }
}

template <int S, bool EDGES>
__global__ void __launch_bounds__(kRowThreads)
k_hist_rows(Grid g, Bins bn, unsigned int *__restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) unsigned int hist[];
  hist_begin(bn, hist);
  unsigned long long bad = 0;
  row_pairs<S>(g, [&](double s, double, double, double, double, double, double) {
    bin_pair<EDGES>(bn, hist, s, bad);
  });
  hist_end(bn, hist, bad, part);
}

__global__ void __launch_bounds__(kRowThreads)
k_scaled_rows(Grid g, SfTable sf, int nsf, double cut2,
             unsigned long long *__restrict__ part) {
  unsigned long long m = 0;
  row_pairs<1>(g, [&](double s, double ax, double ay, double az, double bx, double by, double bz) {
    scaled_pair(sf, nsf, cut2, s, ax, ay, az, bx, by, bz, g.lx, g.ly, g.lz, m);
  });
  mask_end(m, part);
}

// The same on a grid of fewer cells along an axis (long thin boxes): one
// thread per sphere walks the distinct cells of its 27-cell stencil.
template <class F>
__device__ __forceinline__ void sphere_pairs(const Grid &g, int n, F &&f) {
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    const double ax = g.px[p], ay = g.py[p], az = g.pz[p];
    const int cx = search_cell(ax, g.ix, g.nx), cy = search_cell(ay, g.iy, g.ny), cz = search_cell(az, g.iz, g.nz);
    for_stencil(g, cx, cy, cz, [&](int b, int e) {
      for (int q = max(b, p + 1); q < e; ++q) {  // each unordered pair once
        const double bx = g.px[q], by = g.py[q], bz = g.pz[q];
        f(dist2(ax, ay, az, bx, by, bz, g.lx, g.ly, g.lz), ax, ay, az, bx, by, bz);
      }
      return false;
    });
  }
}

template <bool EDGES>
__global__ void __launch_bounds__(256)
k_hist_spheres(Grid g, int n, Bins bn, unsigned int *__restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) unsigned int hist[];
  hist_begin(bn, hist);
  unsigned long long bad = 0;
  sphere_pairs(g, n, [&](double s, double, double, double, double, double, double) {
    bin_pair<EDGES>(bn, hist, s, bad);
  });
  hist_end(bn, hist, bad, part);
}

__global__ void __launch_bounds__(256)
k_scaled_spheres(Grid g, int n, SfTable sf, int nsf, double cut2,
             unsigned long long *__restrict__ part) {
  unsigned long long m = 0;
  sphere_pairs(g, n, [&](double s, double ax, double ay, double az, double bx, double by, double bz) {
    scaled_pair(sf, nsf, cut2, s, ax, ay, az, bx, by, bz, g.lx, g.ly, g.lz, m);
  });
  mask_end(m, part);
}

}  // namespace

namespace hsmc {

long scan_workspace_ints(long n) {
  const long tiles = (n + kScanTile - 1) / kScanTile;
  return 2 * tiles + 1;
}

void exclusive_scan(hipStream_t s, int *in, int n, int *out, int *part, bool clear) {
  if (n == 0) {
    hipLaunchKernelGGL(k_scan_empty, dim3(1), dim3(64), 0, s, out);
    return;
  }
  if (n <= kScanOne) {
    hipLaunchKernelGGL(clear ? k_scan1<true> : k_scan1<false>, dim3(1), dim3(1024), 0, s, in, n, out);
    return;
  }
  const int tiles = (int)(((long)n + kScanTile - 1) / kScanTile);
  int *offs = part + tiles;  // tiles + 1 entries: exclusive offsets and the total
  hipLaunchKernelGGL(clear ? k_scan_tile<true> : k_scan_tile<false>, dim3((unsigned)tiles), dim3(256), 0, s,
                     in, n, out, part);
  hipLaunchKernelGGL(k_scan1<false>, dim3(1), dim3(1024), 0, s, part, tiles, offs);
  hipLaunchKernelGGL(k_scan_add, dim3((unsigned)(((long)n + 255) / 256)), dim3(256), 0, s, out, n, offs, tiles);
}

}  // namespace hsmc

namespace {

int grid_cells_for(double L, double cut) {
  int n = (int)floor(L / cut);
  if (n < 1) n = 1;
  while (n > 1 && L / n < cut) --n;
  return n;
}

// Cells of a search grid of side at least `cut` over a replica's box.
void set_grid(const RepHost &h, double cut, Grid &g) {
  g.nx = grid_cells_for(h.p.lx, cut); g.ny = grid_cells_for(h.p.ly, cut); g.nz = grid_cells_for(h.p.lz, cut);
  g.lx = h.p.lx; g.ly = h.p.ly; g.lz = h.p.lz;
  g.sx = h.p.lx / g.nx; g.sy = h.p.ly / g.ny; g.sz = h.p.lz / g.nz;
  g.ix = 1.0 / g.sx; g.iy = 1.0 / g.sy; g.iz = 1.0 / g.sz;
}

// The C counts of a grid at zero, and in *clear how many of the buffer's are
// once the grid is built: every build's prefix sum leaves the counts it read
// at zero, so only those of a buffer not yet used that far are cleared here.
// Until the build notes *clear (its launches went well), none count as zero.
int clear_counts(hsmc_gpu_ctx *ctx, int *cnt, long C, long *clear) {
  const bool same = ctx->counts_bytes == ctx->scratch_bytes[S_CNT];  // a buffer only ever grows
  const long have = same ? ctx->counts_clear : 0;
  ctx->counts_bytes = ctx->scratch_bytes[S_CNT];
  ctx->counts_clear = 0;
  *clear = std::max(have, C);
  if (have < C) HSMC_HIP(ctx, hipMemsetAsync(cnt + have, 0, sizeof(int) * (C - have), ctx->stream));
  return HSMC_OK;
}

// Build (or reuse) the observable grid of `replica` for cutoff `cut`.
int build_grid(hsmc_gpu_ctx *ctx, int replica, double cut, Grid &g) {
  const RepHost &h = ctx->reps[replica];
  const int N = h.p.n_part;
  set_grid(h, cut, g);
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const long C = (long)nx * ny * nz;
  if (C > (1L << 28)) return HSMC_ERR_NOT_SUPPORTED;
  int *cnt = (int *)scratch(ctx, S_CNT, sizeof(int) * C);
  int *start = (int *)scratch(ctx, S_START, sizeof(int) * (C + 1));
  int2 *cellof = (int2 *)scratch(ctx, S_CELLOF, sizeof(int2) * N);
  int *ids = (int *)scratch(ctx, S_IDS, sizeof(int) * N);
  double *px = (double *)scratch(ctx, S_PX, sizeof(double) * N);
  double *py = (double *)scratch(ctx, S_PY, sizeof(double) * N);
  double *pz = (double *)scratch(ctx, S_PZ, sizeof(double) * N);
  int *part = (int *)scratch(ctx, S_PART, sizeof(int) * scan_workspace_ints(C));
  if (!cnt || !start || !cellof || !ids || !px || !py || !pz || !part)
    return HSMC_ERR_NO_MEMORY;
  g.start = start; g.ids = ids; g.px = px; g.py = py; g.pz = pz;
  if (ctx->aux_replica == replica && ctx->aux_version == ctx->version && ctx->aux_n[0] == nx &&
      ctx->aux_n[1] == ny && ctx->aux_n[2] == nz)
    return HSMC_OK;
  const double *x = ctx->d_x + h.poff, *y = ctx->d_y + h.poff, *z = ctx->d_z + h.poff;
  long clear = 0;
  if (clear_counts(ctx, cnt, C, &clear)) return HSMC_ERR_HIP;
  const unsigned blocks = (unsigned)((N + 255) / 256);
  hipLaunchKernelGGL(k_grid_count<false>, dim3(blocks), dim3(256), 0, ctx->stream, x, y, z, N, nx, ny,
                     nz, g.ix, g.iy, g.iz, cnt, cellof);
  exclusive_scan(ctx->stream, cnt, (int)C, start, part, true);
  hipLaunchKernelGGL(k_grid_scatter, dim3(blocks), dim3(256), 0, ctx->stream, x, y, z, N, cellof,
                     start, ids, px, py, pz);
  HSMC_HIP(ctx, hipGetLastError());
  ctx->counts_clear = clear;
  ctx->aux_replica = replica;
  ctx->aux_version = ctx->version;
  ctx->aux_n[0] = nx; ctx->aux_n[1] = ny; ctx->aux_n[2] = nz;
  ctx->aux_cut = cut;
  return HSMC_OK;
}

constexpr int kWidomLdsSpheres = 2048;
// Above that, or with more cells than 64 KB take, one workgroup of 1024 a
// compute unit files them while grid and positions fit in LDS, the box is not
// so dilute that most of the LDS is empty cells, and filing is not more work
// than the points on a grid that is there already (us a call, grid to be built
// / there / LDS, N = 4000 at density 0.8: 10^5 points 42 / 29 / 31, 10^6 72 /
// 57 / 51, 10^7 302 / 287 / 236; N = 2048 at density 0.3, 2.8 cells a sphere:
// 10^7 661 / 650 / 709).
constexpr size_t kWidomLdsBytes = 158 * 1024;  // and some static words
constexpr long long kWidomLdsPoints = 400000;
constexpr int kSmallRuns = 4096;   // all_pairs: shorter runs for the smallest systems
constexpr double kRowSide = 2.0;   // row_pairs: smallest cell side worth a workgroup

unsigned all_pairs_blocks(int N) {
  const long nt = (N + 63) / 64, waves = (nt + 1) / 2 * (nt + 1) * (N <= kSmallRuns ? 4 : 1);
  return (unsigned)std::min((waves + kPairThreads / 64 - 1) / (kPairThreads / 64), (long)kPairBlocks);
}

// The column sums of the workgroups' rows into the pinned results; above 256
// rows in two steps (1728 rows of 401 counts in one step took 35 us).
int sum_rows(hsmc_gpu_ctx *ctx, const unsigned int *part, int rows, int cols) {
  const dim3 wg(1024);
  const unsigned cb = (unsigned)((cols + 63) / 64);
  if (rows <= 256) {
    hipLaunchKernelGGL(k_sum_rows<unsigned int>, dim3(cb), wg, 0, ctx->stream, part, rows, cols, ctx->h_acc);
  } else {
    const int mid = std::min(64, (rows + 63) / 64);
    unsigned long long *sums = (unsigned long long *)scratch(ctx, S_SUMS, sizeof(unsigned long long) * mid * cols);
    if (!sums) return HSMC_ERR_NO_MEMORY;
    hipLaunchKernelGGL(k_sum_rows<unsigned int>, dim3(cb, mid), wg, 0, ctx->stream, part, rows, cols, sums);
    hipLaunchKernelGGL(k_sum_rows<unsigned long long>, dim3(cb), wg, 0, ctx->stream, sums, mid, cols, ctx->h_acc);
  }
  HSMC_HIP(ctx, hipGetLastError());
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return HSMC_OK;
}

bool cells_at_least(const hsmc_gpu_replica &p, double side, int n) {
  return grid_cells_for(p.lx, side) >= n && grid_cells_for(p.ly, side) >= n &&
         grid_cells_for(p.lz, side) >= n;
}

// First non-negative double at which the monotone condition holds (infinity
// if it holds nowhere), from a guess: usually a few units in the last place
// away, but the bound between "-1" and "above" of a bin width near 1 lies
// anywhere, so the steps double until they pass it and halve from there.
template <class Cond>
double first_double(double guess, Cond &&holds) {
  constexpr long long kInf = 0x7ff0000000000000LL;
  auto at = [&](long long bits) { return holds(__builtin_bit_cast(double, bits)); };
  long long lo = -1, hi = kInf;  // it holds not at lo (below every double) and at hi, or nowhere
  const long long g = std::min(__builtin_bit_cast(long long, guess), kInf);
  for (long long step = 1, p = g; step > 0 && p > lo && p < hi; step *= 2) {
    if (at(p)) {
      hi = p;
      p = g - step;
    } else {
      lo = p;
      p = step < kInf - g ? g + step : kInf;
    }
  }
  while (hi - lo > 1) {
    const long long mid = lo + (hi - lo) / 2;
    (at(mid) ? hi : lo) = mid;
  }
  return __builtin_bit_cast(double, hi);
}

// Edges of the bins (int)((dr - 1.0) / dr_bin) in squared distance, on the
// device: edge[b] is the first s of bin b or later.  Kept by bin width (a
// run bins every sample alike), made longer when more bins are asked for.
int bin_edges(hsmc_gpu_ctx *ctx, double dr_bin, int nbins, const double **edge) {
  double *d = (double *)scratch(ctx, S_BINS, sizeof(double) * (nbins + 1));
  if (!d) return HSMC_ERR_NO_MEMORY;
  if (ctx->edge_bins < nbins || ctx->edge_dr != dr_bin) {
    ctx->edge_bins = 0;  // until they are there
    std::vector<double> e(nbins + 1);
    for (int b = 0; b <= nbins; ++b) {
      const double r = b == 0 ? std::max(0.0, 1.0 - dr_bin) : 1.0 + b * dr_bin;
      // truncation towards zero puts quotients in (-1, 0) in bin 0
      e[b] = first_double(r * r, [&](double s) {
        const double q = (sqrt(s) - 1.0) / dr_bin;
        return b == 0 ? q > -1.0 : q >= (double)b;
      });
    }
    HSMC_HIP(ctx, hipMemcpyAsync(d, e.data(), sizeof(double) * (nbins + 1), hipMemcpyHostToDevice, ctx->stream));
    HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    ctx->edge_dr = dr_bin;
    ctx->edge_bins = nbins;
  }
  *edge = d;
  return HSMC_OK;
}

bool bad_replica(const hsmc_gpu_ctx *ctx, int r) { return !ctx || r < 0 || r >= ctx->R; }

__global__ void k_zero_words(unsigned int *__restrict__ p, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Workspace layout of the scan: counts and starts of the grid's C cells, cell
// (and place in it) of the N spheres and their sorted positions, each region
// 256-B aligned; 32 bytes a sphere and 12 a cell.  The workgroups' result masks
// lie over the cells, which are read no more once the spheres are sorted.
struct ScanLayout {
  size_t cnt, start, cellof, px, py, pz, part, bytes;
};

ScanLayout scan_layout(long N, long C) {
  ScanLayout l{};
  size_t o = 0;
  auto take = [&](size_t b) {
    const size_t at = o;
    o += align256(b);
    return at;
  };
  l.cnt = take(sizeof(int) * C);
  l.start = take(sizeof(int) * (C + 1));
  l.cellof = take(sizeof(int2) * N);
  l.px = take(sizeof(double) * N);
  l.py = take(sizeof(double) * N);
  l.pz = take(sizeof(double) * N);
  l.part = take(sizeof(int) * scan_workspace_ints(C));
  // room this build does without (a second count of the cells, the scale table
  // and a mask): the size asked for, and so the call that is refused, stays
  take(sizeof(int) * C);
  take(sizeof(double) * 64);
  take(sizeof(unsigned long long));
  l.bytes = o;
  return l;
}

int scan_cut(const double *sf, int n_sf, double *cut) {
  double smin = 1.0;
  for (int k = 0; k < n_sf; ++k) {
    if (!(sf[k] > 0.0)) return HSMC_ERR_BAD_ARG;
    smin = std::min(smin, sf[k]);
  }
  *cut = (1.0 / smin) * (1.0 + 1e-6);
  return HSMC_OK;
}

}  // namespace

namespace hsmc {

size_t overlap_scan_workspace_bytes(const hsmc_gpu_ctx *ctx, int replica, const double *sf, int n_sf) {
  if (bad_replica(ctx, replica) || n_sf < 1 || n_sf > 64 || !sf) return 0;
  double cut = 0.0;
  if (scan_cut(sf, n_sf, &cut)) return 0;
  const hsmc_gpu_replica &p = ctx->reps[replica].p;
  const long C = (long)grid_cells_for(p.lx, cut) * grid_cells_for(p.ly, cut) * grid_cells_for(p.lz, cut);
  return scan_layout(p.n_part, C).bytes;
}

// The scan of hsmc_gpu_any_overlap_scaled with every buffer carved from the
// device workspace ws (ws_bytes long): the same kernels, the grid rebuilt from
// the replica's positions, counters cleared by kernels, the scale factors
// passed by value.  Nothing is allocated.
int overlap_scan_in_workspace(hsmc_gpu_ctx *ctx, int replica, const double *sf, int n_sf,
                              unsigned char *ws, size_t ws_bytes, uint8_t *no_overlap) {
  if (bad_replica(ctx, replica) || n_sf < 1 || n_sf > 64 || !sf || !no_overlap || !ws)
    return HSMC_ERR_BAD_ARG;
  double cut = 0.0;
  int st = scan_cut(sf, n_sf, &cut);
  if (st) return st;
  const RepHost &h = ctx->reps[replica];
  const int N = h.p.n_part;
  Grid g;
  set_grid(h, cut, g);
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const long C = (long)nx * ny * nz;
  const ScanLayout l = scan_layout(N, C);
  if (l.bytes > ws_bytes) {
    ctx->last_error = "the scan needs " + std::to_string(l.bytes) + " bytes of workspace, " +
                      std::to_string(ws_bytes) + " available";
    return HSMC_ERR_NOT_SUPPORTED;
  }
  int *cnt = (int *)(ws + l.cnt), *start = (int *)(ws + l.start);
  int2 *cellof = (int2 *)(ws + l.cellof);
  double *px = (double *)(ws + l.px), *py = (double *)(ws + l.py), *pz = (double *)(ws + l.pz);
  unsigned long long *dmask = (unsigned long long *)(ws + l.cellof);
  g.start = start; g.ids = nullptr; g.px = px; g.py = py; g.pz = pz;
  const long zero_words = C;
  hipLaunchKernelGGL(k_zero_words, dim3((unsigned)((zero_words + 255) / 256)), dim3(256), 0, ctx->stream,
                     (unsigned int *)cnt, zero_words);
  SfTable t{};
  for (int k = 0; k < n_sf; ++k) t.v[k] = sf[k];
  const double *x = ctx->d_x + h.poff, *y = ctx->d_y + h.poff, *z = ctx->d_z + h.poff;
  const unsigned blocks = (unsigned)((N + 255) / 256);
  hipLaunchKernelGGL(k_grid_count<false>, dim3(blocks), dim3(256), 0, ctx->stream, x, y, z, N, nx, ny,
                     nz, g.ix, g.iy, g.iz, cnt, cellof);
  exclusive_scan(ctx->stream, cnt, (int)C, start, (int *)(ws + l.part), false);
  hipLaunchKernelGGL(k_grid_scatter, dim3(blocks), dim3(256), 0, ctx->stream, x, y, z, N, cellof,
                     start, (int *)nullptr, px, py, pz);
  hipLaunchKernelGGL(k_scaled_spheres, dim3(blocks), dim3(256), 0, ctx->stream, g, N, t, n_sf,
                     cut * cut, dmask);
  hipLaunchKernelGGL(k_sum_all<true>, dim3(1), dim3(1024), 0, ctx->stream, dmask, (int)blocks,
                     (const unsigned *)nullptr, ctx->h_acc);
  HSMC_HIP(ctx, hipGetLastError());
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  const unsigned long long mask = ctx->h_acc[0];
  for (int k = 0; k < n_sf; ++k) no_overlap[k] = ((mask >> k) & 1ull) ? 0 : 1;
  return HSMC_OK;
}

}  // namespace hsmc

extern "C" {

int hsmc_gpu_cell_list(hsmc_gpu_ctx *ctx, int replica, int nx, int ny, int nz, int max_part,
                       int32_t *part_cell, int32_t *neigh_mat) {
  if (bad_replica(ctx, replica) || nx < 1 || ny < 1 || nz < 1 || max_part < 2)
    return HSMC_ERR_BAD_ARG;
  const RepHost &h = ctx->reps[replica];
  const double sx = h.p.lx / nx, sy = h.p.ly / ny, sz = h.p.lz / nz;
  if (sx < 1.0 || sy < 1.0 || sz < 1.0) return HSMC_ERR_CELL_TOO_SMALL;  // cell_list.c:126-129
  const long C = (long)nx * ny * nz;
  const int N = h.p.n_part;
  if (part_cell) {
    int *cnt = (int *)scratch(ctx, S_CNT, sizeof(int) * C);
    int *start = (int *)scratch(ctx, S_START, sizeof(int) * (C + 1));
    int2 *cellof = (int2 *)scratch(ctx, S_CELLOF, sizeof(int2) * N);
    int *ids = (int *)scratch(ctx, S_IDS, sizeof(int) * N);
    double *px = (double *)scratch(ctx, S_PX, sizeof(double) * N);
    double *py = (double *)scratch(ctx, S_PY, sizeof(double) * N);
    double *pz = (double *)scratch(ctx, S_PZ, sizeof(double) * N);
    int *rows = (int *)scratch(ctx, S_OUT0, sizeof(int) * C * max_part);
    int *part = (int *)scratch(ctx, S_PART, sizeof(int) * scan_workspace_ints(C));
    if (!cnt || !start || !cellof || !ids || !px || !py || !pz || !rows || !part)
      return HSMC_ERR_NO_MEMORY;
    ctx->aux_replica = -1;  // the CSR scratch now holds this grid
    const double *x = ctx->d_x + h.poff, *y = ctx->d_y + h.poff, *z = ctx->d_z + h.poff;
    long clear = 0;
    if (clear_counts(ctx, cnt, C, &clear)) return HSMC_ERR_HIP;
    const unsigned blocks = (unsigned)((N + 255) / 256);
    hipLaunchKernelGGL(k_grid_count<true>, dim3(blocks), dim3(256), 0, ctx->stream, x, y, z, N, nx, ny,
                       nz, sx, sy, sz, cnt, cellof);
    exclusive_scan(ctx->stream, cnt, (int)C, start, part, true);
    hipLaunchKernelGGL(k_grid_scatter, dim3(blocks), dim3(256), 0, ctx->stream, x, y, z, N, cellof,
                     start, ids, px, py, pz);
    hipLaunchKernelGGL(k_part_cell, dim3((unsigned)((C + 255) / 256)), dim3(256), 0, ctx->stream,
                       start, (int)C, ids, max_part, rows, ctx->d_err);
    HSMC_HIP(ctx, hipGetLastError());
    ctx->counts_clear = clear;
    HSMC_HIP(ctx, hipMemcpyAsync(part_cell, rows, sizeof(int) * C * max_part,
                                 hipMemcpyDeviceToHost, ctx->stream));
    HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    int st = check_device_errors(ctx);
    if (st) return st;
  }
  if (neigh_mat) {  // neigh_id (cell_list.c:266-301), host-side table
    for (int a = 0; a < nx; ++a)
      for (int b = 0; b < ny; ++b)
        for (int c = 0; c < nz; ++c) {
          const long ref = ((long)a * ny + b) * nz + c;
          int counter = 0;
          for (int i = -1; i < 2; ++i)
            for (int j = -1; j < 2; ++j)
              for (int k = -1; k < 2; ++k) {
                int ix = a + i, iy = b + j, iz = c + k;
                if (ix > nx - 1) ix -= nx; else if (ix < 0) ix += nx;
                if (iy > ny - 1) iy -= ny; else if (iy < 0) iy += ny;
                if (iz > nz - 1) iz -= nz; else if (iz < 0) iz += nz;
                neigh_mat[ref * 27 + counter] = (ix * ny + iy) * nz + iz;
                ++counter;
              }
        }
  }
  return HSMC_OK;
}

int hsmc_gpu_overlap_batch(hsmc_gpu_ctx *ctx, int replica, const int32_t *idx, const double *xyz,
                           int m, uint8_t *out) {
  if (bad_replica(ctx, replica) || m < 0 || (m > 0 && (!idx || !xyz || !out))) return HSMC_ERR_BAD_ARG;
  if (m == 0) return HSMC_OK;
  for (int k = 0; k < m; ++k)
    if (idx[k] < 0 || idx[k] >= ctx->reps[replica].p.n_part) return HSMC_ERR_BAD_ARG;
  const RepHost &h = ctx->reps[replica];
  // (a point outside the box meets only the cells beside its own on a grid)
  bool few = m <= kFewQueries && h.p.n_part <= kFewSpheres;
  FewQueries f{};
  const double L[3] = {h.p.lx, h.p.ly, h.p.lz};
  for (int k = 0; few && k < m; ++k) {
    for (int a = 0; a < 3; ++a) {
      f.q[k][a] = xyz[3 * k + a];
      few = few && f.q[k][a] >= 0.0 && f.q[k][a] <= L[a];
    }
    f.idx[k] = idx[k];
  }
  if (few) {
    hipLaunchKernelGGL(k_overlap_few, dim3((unsigned)m), dim3(1024), 0, ctx->stream, f, ctx->d_x + h.poff,
                       ctx->d_y + h.poff, ctx->d_z + h.poff, h.p.n_part, h.p.lx, h.p.ly, h.p.lz, ctx->h_acc);
    HSMC_HIP(ctx, hipGetLastError());
    HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    for (int k = 0; k < m; ++k) out[k] = (uint8_t)ctx->h_acc[k];
    return HSMC_OK;
  }
  Grid g;
  int st = build_grid(ctx, replica, 1.0 + 1e-9, g);
  if (st) return st;
  int *didx = (int *)scratch(ctx, S_Q0, sizeof(int) * m);
  double *dq = (double *)scratch(ctx, S_Q1, sizeof(double) * 3 * m);
  unsigned char *dout = (unsigned char *)scratch(ctx, S_Q2, m);
  if (!didx || !dq || !dout) return HSMC_ERR_NO_MEMORY;
  HSMC_HIP(ctx, hipMemcpyAsync(didx, idx, sizeof(int) * m, hipMemcpyHostToDevice, ctx->stream));
  HSMC_HIP(ctx, hipMemcpyAsync(dq, xyz, sizeof(double) * 3 * m, hipMemcpyHostToDevice, ctx->stream));
  hipLaunchKernelGGL(k_overlap_batch, dim3((m + 255) / 256), dim3(256), 0, ctx->stream, g, didx, dq,
                     m, dout);
  HSMC_HIP(ctx, hipGetLastError());
  HSMC_HIP(ctx, hipMemcpyAsync(out, dout, m, hipMemcpyDeviceToHost, ctx->stream));
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return HSMC_OK;
}

int hsmc_gpu_overlap_scaled(hsmc_gpu_ctx *ctx, int replica, const int32_t *idx, const double *sf,
                            int m, uint8_t *out) {
  if (bad_replica(ctx, replica) || m < 0 || (m > 0 && (!idx || !sf || !out))) return HSMC_ERR_BAD_ARG;
  if (m == 0) return HSMC_OK;
  double smin = 1.0;
  for (int k = 0; k < m; ++k) {
    if (idx[k] < 0 || idx[k] >= ctx->reps[replica].p.n_part || !(sf[k] > 0.0)) return HSMC_ERR_BAD_ARG;
    smin = std::min(smin, sf[k]);
  }
  Grid g;
  int st = build_grid(ctx, replica, (1.0 / smin) * (1.0 + 1e-9), g);
  if (st) return st;
  const RepHost &h = ctx->reps[replica];
  int *didx = (int *)scratch(ctx, S_Q0, sizeof(int) * m);
  double *dsf = (double *)scratch(ctx, S_Q1, sizeof(double) * m);
  unsigned char *dout = (unsigned char *)scratch(ctx, S_Q2, m);
  if (!didx || !dsf || !dout) return HSMC_ERR_NO_MEMORY;
  HSMC_HIP(ctx, hipMemcpyAsync(didx, idx, sizeof(int) * m, hipMemcpyHostToDevice, ctx->stream));
  HSMC_HIP(ctx, hipMemcpyAsync(dsf, sf, sizeof(double) * m, hipMemcpyHostToDevice, ctx->stream));
  hipLaunchKernelGGL(k_overlap_scaled, dim3((m + 255) / 256), dim3(256), 0, ctx->stream, g,
                     ctx->d_x + h.poff, ctx->d_y + h.poff, ctx->d_z + h.poff, didx, dsf, m, dout);
  HSMC_HIP(ctx, hipGetLastError());
  HSMC_HIP(ctx, hipMemcpyAsync(out, dout, m, hipMemcpyDeviceToHost, ctx->stream));
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return HSMC_OK;
}

int hsmc_gpu_any_overlap_scaled(hsmc_gpu_ctx *ctx, int replica, const double *sf, int n_sf,
                                uint8_t *no_overlap) {
  if (bad_replica(ctx, replica) || n_sf < 1 || n_sf > 64 || !sf || !no_overlap) return HSMC_ERR_BAD_ARG;
  double smin = 1.0;
  for (int k = 0; k < n_sf; ++k) {
    if (!(sf[k] > 0.0)) return HSMC_ERR_BAD_ARG;
    smin = std::min(smin, sf[k]);
  }
  const double cut = (1.0 / smin) * (1.0 + 1e-6), cut2 = cut * cut;
  const RepHost &h = ctx->reps[replica];
  const int N = h.p.n_part;
  SfTable t{};
  for (int k = 0; k < n_sf; ++k) t.v[k] = sf[k];
  unsigned blocks;
  unsigned long long *part;
  if (N <= kAllPairs) {
    const double *x = ctx->d_x + h.poff, *y = ctx->d_y + h.poff, *z = ctx->d_z + h.poff;
    blocks = all_pairs_blocks(N);
    part = (unsigned long long *)scratch(ctx, S_OUT0, sizeof(unsigned long long) * blocks);
    if (!part) return HSMC_ERR_NO_MEMORY;
    hipLaunchKernelGGL(N <= kSmallRuns ? k_scaled_all<16> : k_scaled_all<64>, dim3(blocks),
                       dim3(kPairThreads), 0, ctx->stream, x, y, z, N, h.p.lx, h.p.ly, h.p.lz, t, n_sf,
                       cut2, part);
  } else {
    // cells of a few spheres give row_pairs' lanes work
    const double side = std::max(cut, kRowSide);
    const bool rows = cells_at_least(h.p, side, 3);
    Grid g;
    int st = build_grid(ctx, replica, rows ? side : cut, g);
    if (st) return st;
    const long C = (long)g.nx * g.ny * g.nz;
    blocks = (unsigned)std::min(rows ? C : ((long)N + 255) / 256, (long)kRowBlocks);
    part = (unsigned long long *)scratch(ctx, S_OUT0, sizeof(unsigned long long) * blocks);
    if (!part) return HSMC_ERR_NO_MEMORY;
    if (rows)
      hipLaunchKernelGGL(k_scaled_rows, dim3(blocks), dim3(kRowThreads), 0, ctx->stream, g, t, n_sf,
                         cut2, part);
    else
      hipLaunchKernelGGL(k_scaled_spheres, dim3(blocks), dim3(256), 0, ctx->stream, g, N, t, n_sf, cut2,
                         part);
  }
  hipLaunchKernelGGL(k_sum_all<true>, dim3(1), dim3(1024), 0, ctx->stream, part, (int)blocks,
                     (const unsigned *)nullptr, ctx->h_acc);
  HSMC_HIP(ctx, hipGetLastError());
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  const unsigned long long mask = ctx->h_acc[0];
  for (int k = 0; k < n_sf; ++k) no_overlap[k] = ((mask >> k) & 1ull) ? 0 : 1;
  return HSMC_OK;
}

int hsmc_gpu_pair_dist(hsmc_gpu_ctx *ctx, int replica, const int32_t *i, const int32_t *j, int m,
                       double sf, double *out) {
  if (bad_replica(ctx, replica) || m < 0 || (m > 0 && (!i || !j || !out)) || !(sf > 0.0))
    return HSMC_ERR_BAD_ARG;
  if (m == 0) return HSMC_OK;
  const RepHost &h = ctx->reps[replica];
  for (int k = 0; k < m; ++k)
    if (i[k] < 0 || i[k] >= h.p.n_part || j[k] < 0 || j[k] >= h.p.n_part) return HSMC_ERR_BAD_ARG;
  int *di = (int *)scratch(ctx, S_Q0, sizeof(int) * m);
  int *dj = (int *)scratch(ctx, S_Q2, sizeof(int) * m);
  double *dout = (double *)scratch(ctx, S_Q1, sizeof(double) * m);
  if (!di || !dj || !dout) return HSMC_ERR_NO_MEMORY;
  HSMC_HIP(ctx, hipMemcpyAsync(di, i, sizeof(int) * m, hipMemcpyHostToDevice, ctx->stream));
  HSMC_HIP(ctx, hipMemcpyAsync(dj, j, sizeof(int) * m, hipMemcpyHostToDevice, ctx->stream));
  hipLaunchKernelGGL(k_pair_dist, dim3((m + 255) / 256), dim3(256), 0, ctx->stream,
                     ctx->d_x + h.poff, ctx->d_y + h.poff, ctx->d_z + h.poff, di, dj, m, sf,
                     h.p.lx, h.p.ly, h.p.lz, dout);
  HSMC_HIP(ctx, hipGetLastError());
  HSMC_HIP(ctx, hipMemcpyAsync(out, dout, sizeof(double) * m, hipMemcpyDeviceToHost, ctx->stream));
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return HSMC_OK;
}

static int pair_hist(hsmc_gpu_ctx *ctx, int replica, double dr_bin, int nbins, double rmax_eff,
                     int64_t *counts, int64_t *oor) {
  if (bad_replica(ctx, replica) || !(dr_bin > 0.0) || nbins < 1 || nbins > 8192 ||
      !(rmax_eff > 1.0) || !counts)
    return HSMC_ERR_BAD_ARG;
  const RepHost &h = ctx->reps[replica];
  const double half = std::min(h.p.lx, std::min(h.p.ly, h.p.lz)) / 2.0;
  if (rmax_eff > half * (1.0 + 1e-12)) {
    ctx->last_error = "histogram cutoff beyond half the box (minimum image)";
    return HSMC_ERR_BAD_ARG;
  }
  const double cut = rmax_eff * (1.0 + 1e-9);
  const int N = h.p.n_part;
  Bins bn{dr_bin, rmax_eff, 0.0, (float)(1.0 / dr_bin), nbins, nullptr};
  bn.smax = first_double(rmax_eff * rmax_eff, [&](double s) { return !(sqrt(s) < rmax_eff); });
  // the edges for the many bins of g(r); a contact histogram's few pairs are
  // binned by the formula, and above 2048 bins the edges would leave LDS
  const bool edges = nbins > 16 && nbins <= 2048;
  if (edges) {
    int st = bin_edges(ctx, dr_bin, nbins, &bn.edge);
    if (st) return st;
  }
  const size_t lds = sizeof(unsigned int) * (((size_t)nbins + 1) & ~(size_t)1) +
                     (edges ? sizeof(double) * ((size_t)nbins + 1) : 0);
  unsigned blocks;
  auto rows_of = [&]() {
    return (unsigned int *)scratch(ctx, S_OUT0, sizeof(unsigned int) * ((size_t)nbins + 2) * blocks);
  };
  unsigned int *part;
  if (N <= (rmax_eff < kWide ? kAllPairs : kAllPairsWide)) {
    const double *x = ctx->d_x + h.poff, *y = ctx->d_y + h.poff, *z = ctx->d_z + h.poff;
    blocks = all_pairs_blocks(N);
    part = rows_of();
    if (!part) return HSMC_ERR_NO_MEMORY;
    auto fn = N <= kSmallRuns ? (edges ? k_hist_all<16, true> : k_hist_all<16, false>)
                              : (edges ? k_hist_all<64, true> : k_hist_all<64, false>);
    hipLaunchKernelGGL(fn, dim3(blocks), dim3(kPairThreads), lds, ctx->stream, x, y, z, N, h.p.lx,
                       h.p.ly, h.p.lz, bn, part);
  } else {
    // a stencil of 5^3 cells of half the cutoff has 0.58 of the volume of
    // 3^3 cells of the cutoff, as long as those cells hold some spheres
    const bool two = rmax_eff >= kWide && cells_at_least(h.p, cut / 2.0, 5);
    const double side = two ? cut / 2.0 : std::max(cut, kRowSide);
    const bool rows = two || cells_at_least(h.p, side, 3);
    Grid g;
    int st = build_grid(ctx, replica, rows ? side : cut, g);
    if (st) return st;
    const long C = (long)g.nx * g.ny * g.nz;
    blocks = (unsigned)std::min(rows ? C : ((long)N + 255) / 256, (long)kRowBlocks);
    part = rows_of();
    if (!part) return HSMC_ERR_NO_MEMORY;
    if (rows) {
      auto fn = two ? (edges ? k_hist_rows<2, true> : k_hist_rows<2, false>)
                    : (edges ? k_hist_rows<1, true> : k_hist_rows<1, false>);
      hipLaunchKernelGGL(fn, dim3(blocks), dim3(kRowThreads), lds, ctx->stream, g, bn, part);
    } else {
      hipLaunchKernelGGL(edges ? k_hist_spheres<true> : k_hist_spheres<false>, dim3(blocks), dim3(256),
                         lds, ctx->stream, g, N, bn, part);
    }
  }
  HSMC_HIP(ctx, hipGetLastError());
  int st = sum_rows(ctx, part, (int)blocks, nbins + 2);
  if (st) return st;
  for (int b = 0; b < nbins; ++b) counts[b] = (int64_t)ctx->h_acc[b];
  if (oor) *oor = (int64_t)(ctx->h_acc[nbins] + (ctx->h_acc[nbins + 1] << 32));
  return HSMC_OK;
}

int hsmc_gpu_rdf_counts(hsmc_gpu_ctx *ctx, int replica, double dr_bin, int nbins, double rmax_eff,
                        int64_t *counts, int64_t *out_of_range) {
  return pair_hist(ctx, replica, dr_bin, nbins, rmax_eff, counts, out_of_range);
}

int hsmc_gpu_contact_counts(hsmc_gpu_ctx *ctx, int replica, double dr_bin, int nbins,
                            double rmax_eff, int64_t *counts, int64_t *out_of_range) {
  return pair_hist(ctx, replica, dr_bin, nbins, rmax_eff, counts, out_of_range);
}

int hsmc_gpu_widom_points(hsmc_gpu_ctx *ctx, int replica, const double *xyz, int m, uint8_t *hit,
                          int64_t *hits) {
  if (bad_replica(ctx, replica) || m < 0 || (m > 0 && !xyz)) return HSMC_ERR_BAD_ARG;
  if (m == 0) {
    if (hits) *hits = 0;
    return HSMC_OK;
  }
  Grid g;
  int st = build_grid(ctx, replica, 1.0 + 1e-9, g);
  if (st) return st;
  double *dq = (double *)scratch(ctx, S_Q1, sizeof(double) * 3 * m);
  unsigned char *dout = (unsigned char *)scratch(ctx, S_Q2, m);
  if (!dq || !dout) return HSMC_ERR_NO_MEMORY;
  HSMC_HIP(ctx, hipMemcpyAsync(dq, xyz, sizeof(double) * 3 * m, hipMemcpyHostToDevice, ctx->stream));
  hipLaunchKernelGGL(k_widom_points, dim3((m + 255) / 256), dim3(256), 0, ctx->stream, g, dq, m, dout);
  HSMC_HIP(ctx, hipGetLastError());
  std::vector<uint8_t> tmp;
  uint8_t *dst = hit;
  if (!dst) {
    tmp.resize(m);
    dst = tmp.data();
  }
  HSMC_HIP(ctx, hipMemcpyAsync(dst, dout, m, hipMemcpyDeviceToHost, ctx->stream));
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (hits) {
    int64_t s = 0;
    for (int k = 0; k < m; ++k) s += dst[k];
    *hits = s;
  }
  return HSMC_OK;
}

int hsmc_gpu_widom_uniform(hsmc_gpu_ctx *ctx, int replica, uint64_t seed, uint64_t sample,
                           int64_t first, int64_t n, int64_t *hits) {
  if (bad_replica(ctx, replica) || n < 0 || first < 0 || !hits) return HSMC_ERR_BAD_ARG;
  *hits = 0;
  if (n == 0) return HSMC_OK;
  const RepHost &h = ctx->reps[replica];
  const int N = h.p.n_part;
  Grid g;
  set_grid(h, 1.0 + 1e-9, g);
  const size_t lds = widom_lds_bytes(N, (long)g.nx * g.ny * g.nz);
  const bool small = N <= kWidomLdsSpheres && lds <= 64 * 1024;
  const bool kept = ctx->aux_replica == replica && ctx->aux_version == ctx->version && ctx->aux_n[0] == g.nx &&
                    ctx->aux_n[1] == g.ny && ctx->aux_n[2] == g.nz;
  const bool in_lds = small || (lds <= kWidomLdsBytes && (long)g.nx * g.ny * g.nz <= 2L * N &&
                                !(kept && n < kWidomLdsPoints));
  const long long wg = in_lds ? (small ? kWidomLdsThreads : 1024) : 256;
  const long long most = in_lds ? (small ? kWidomLdsBlocks : ctx->n_cu) : kWidomUniformBlocks;
  const long long blocks = std::min((n + wg - 1) / wg, most);
  unsigned long long *part = (unsigned long long *)scratch(ctx, S_OUT0, sizeof(unsigned long long) * blocks);
  if (!part) return HSMC_ERR_NO_MEMORY;
  if (in_lds) {
    auto fn = small ? k_widom_uniform_lds<kWidomLdsThreads> : k_widom_uniform_lds<1024>;
    if (lds > 64 * 1024)  // always the same value: contexts of other threads launch this kernel too
      HSMC_HIP(ctx, hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kWidomLdsBytes));
    hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3((unsigned)wg), lds, ctx->stream, g, N,
                       ctx->d_x + h.poff, ctx->d_y + h.poff, ctx->d_z + h.poff, (uint32_t)seed,
                       (uint32_t)(seed >> 32), (unsigned long long)sample, (long long)first, (long long)n, part);
  } else {
    int st = build_grid(ctx, replica, 1.0 + 1e-9, g);
    if (st) return st;
    hipLaunchKernelGGL(k_widom_uniform, dim3((unsigned)blocks), dim3((unsigned)wg), 0, ctx->stream, g,
                       (uint32_t)seed, (uint32_t)(seed >> 32), (unsigned long long)sample,
                       (long long)first, (long long)n, part);
  }
  hipLaunchKernelGGL(k_sum_all<false>, dim3(1), dim3(1024), 0, ctx->stream, part, (int)blocks,
                     (const unsigned *)nullptr, ctx->h_acc);
  HSMC_HIP(ctx, hipGetLastError());
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  *hits = (int64_t)ctx->h_acc[0];
  return HSMC_OK;
}

int hsmc_gpu_widom_cells(hsmc_gpu_ctx *ctx, int replica, uint64_t seed, uint64_t sample,
                         int32_t per_cell, int64_t *hits, int64_t *n_points, int32_t out_grid[3]) {
  if (bad_replica(ctx, replica) || per_cell < 0 || !hits) return HSMC_ERR_BAD_ARG;
  *hits = 0;
  Grid g;
  int st = build_grid(ctx, replica, 1.0 + 1e-9, g);
  if (st) return st;
  const long C = (long)g.nx * g.ny * g.nz;
  if (n_points) *n_points = (int64_t)per_cell * C;
  if (out_grid) {
    out_grid[0] = g.nx;
    out_grid[1] = g.ny;
    out_grid[2] = g.nz;
  }
  if (per_cell == 0) return HSMC_OK;
  // spheres of unit diameter centred in a 27-cell stencil fit in a box one
  // diameter wider: at most the close-packing fraction (0.7405, taken as
  // 0.78) of its volume over the sphere volume
  const double span = (std::min(3, g.nx) * g.sx + 1.0) * (std::min(3, g.ny) * g.sy + 1.0) *
                      (std::min(3, g.nz) * g.sz + 1.0);
  const long bound = std::min((long)ctx->reps[replica].p.n_part, (long)ceil(0.78 * span / (M_PI / 6.0)));
  if (bound > kWidomCellsLcap) {
    ctx->last_error = "observable-grid cells too wide for the stratified insertion kernel";
    return HSMC_ERR_NOT_SUPPORTED;
  }
  const long blocks = std::min((C + kWidomCellsWaves - 1) / kWidomCellsWaves, (long)kWidomCellsBlocks);
  unsigned long long *part = (unsigned long long *)scratch(ctx, S_OUT0, sizeof(unsigned long long) * blocks);
  if (!part) return HSMC_ERR_NO_MEMORY;
  const bool fast = g.nx >= 3 && g.ny >= 3 && g.nz >= 3;
  hipLaunchKernelGGL(fast ? k_widom_cells<true> : k_widom_cells<false>, dim3((unsigned)blocks), dim3(64 * kWidomCellsWaves), 0, ctx->stream, g,
                     (uint32_t)seed, (uint32_t)(seed >> 32), (unsigned long long)sample, (int)per_cell,
                     part, ctx->d_err);
  hipLaunchKernelGGL(k_sum_all<false>, dim3(1), dim3(1024), 0, ctx->stream, part, (int)blocks, ctx->d_err,
                     ctx->h_acc);
  HSMC_HIP(ctx, hipGetLastError());
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  *hits = (int64_t)ctx->h_acc[0];
  return ctx->h_acc[1] ? check_device_errors(ctx) : HSMC_OK;  // the kernel's view of the sticky bits
}

}  // extern "C"
