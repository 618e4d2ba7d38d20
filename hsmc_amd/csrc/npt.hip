// npt.hip -- isobaric (NpT) sweeps of many replicas at once.
//
// A sweep of the reference's NpT chain (sweep_npt, npt.c:177-196) makes N
// steps, each a volume move with probability 1/(N+1) (npt.c:185).  Here a
// sweep is one checkerboard particle sweep of every replica followed by each
// replica's Binomial(N, 1/(N+1)) volume moves (vol_move, moves.c:83-153):
//   ln V' = ln V + (r - 0.5) dv_max,  sf = (V'/V)^(1/3);
//   rejected if any pair overlaps after scaling every coordinate and the box
//   by sf (moves.c:104-112); else accepted when
//   r' < exp(-beta P (V' - V) + (N + 1) ln(V'/V)) (moves.c:117-121), and then
//   positions and box are scaled by sf (moves.c:129-142).
// Both kernels leave the NpT distribution invariant, so their composition
// samples it.  In rounds, round t holds the t-th move of every replica that
// draws more than t, and one kernel checks every compression of the round.
//
// Small replicas make all of a sweep's moves in one launch (k_volume_moves;
// moves_in_one_launch says which), others round by round with the scan below.
//
// That scan reads the cell list the last sweep left (the sweep grid: cells of
// side > 1 holding every sphere, filed by the sweep's rebin and kept by its
// moves, none of which leaves its cell).  A pair closer than 1/sf before
// scaling lies in neighbouring cells whenever the cell side is at least 1/sf,
// which holds for the small volume steps NpT runs use; a replica whose cells
// are narrower falls back to the single-replica scan on a grid of side 1/sf.
//
// Each replica's volume draws come from a host Philox4x32-10 stream keyed by
// its seed (counter: sweep, round, 0, "NPT\0"), so its run does not depend
// on the other replicas of the batch.
#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "ctx.h"
#include "device_common.h"

using namespace hsmc;

namespace {

constexpr int S_FLAG = 15, S_BLK = 16, S_MOVE = 17;  // context scratch slots
constexpr uint32_t kNptTag = 0x4E505400u;  // "NPT\0"

// Any pair of a replica with a proposed compression (sf[r] > 0) closer than 1
// after scaling: thread per sphere, neighbours from the last sweep's cells.
// Blocks cover only the replicas that propose a compression: block b takes
// the 256 spheres from blk[b] on, all of one replica, so the replica (and
// its record) is uniform and the block stops as a whole once the replica
// has an overlap.
// Each pair is tested once: from the sphere's own cell towards the 13
// lexicographically forward neighbour cells, and within the cell towards
// higher ids (the scaled distance is the same from either end, as
// fl(a - b) = -fl(b - a)).  A thread stops once its replica has an overlap.
__global__ void __launch_bounds__(256)
k_vol_overlap(const RepDev *__restrict__ reps, const SweepDev *__restrict__ swp, int R,
              const int *__restrict__ prep, const int *__restrict__ blk, int C,
              const int *__restrict__ cnt, const SlotRec *__restrict__ slot_all, int cap,
              const unsigned long long *__restrict__ sweep_next, const double *__restrict__ x,
              const double *__restrict__ y, const double *__restrict__ z,
              const double *__restrict__ sfr, int *__restrict__ flags) {
  const int i0 = blk[blockIdx.x];
  const int r = prep[i0];
  const RepDev rp = reps[r];
  const int i = i0 + (int)threadIdx.x;
  if (i >= rp.poff + rp.N) return;
  const double sf = sfr[r];
  if (!(sf > 0.0)) return;  // the whole block
  if (__hip_atomic_load(&flags[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  const unsigned long long sweep = *sweep_next - 1ull;
  const int *cntb = cnt + (size_t)(sweep & 1ull) * C;
  // one replica keeps slot records and table entries per sweep parity
  const int sb = R == 1 ? (int)(sweep & 1ull) : 0;
  const SlotRec *slot = slot_all + (size_t)sb * cap * C;
  // the last sweep's grid shift, as its rebin drew it (swp points at the
  // last sweep's entry when there is one replica)
  const double shx = swp[r].shx, shy = swp[r].shy, shz = swp[r].shz;
  const double ax = x[i], ay = y[i], az = z[i];
  const int cx = filed_cell(ax, shx, rp.lx, rp.ix, rp.gx);
  const int cy = filed_cell(ay, shy, rp.ly, rp.iy, rp.gy);
  const int cz = filed_cell(az, shz, rp.lz, rp.iz, rp.gz);
  const int me = i - rp.poff;
  // d = 13 is the own cell; d = 14..26 are the forward offsets.  The
  // answer does not depend on the order of the tests, so the 14 cells'
  // counts load together, and each cell's first two slots load with the
  // poll of the replica's flag (an overlap found elsewhere ends the scan).
  int cell[14], n[14];
#pragma unroll
  for (int j = 0; j < 14; ++j) {
    const int d = 13 + j;
    const int dx = d / 9 - 1, dy = (d / 3) % 3 - 1, dz = d % 3 - 1;
    const bool ok = stencil_axis_ok(dx, rp.gx) && stencil_axis_ok(dy, rp.gy) && stencil_axis_ok(dz, rp.gz);
    cell[j] = rp.coff + (ok ? (wrap_index(cx + dx, rp.gx) * rp.gy + wrap_index(cy + dy, rp.gy)) * rp.gz +
                                  wrap_index(cz + dz, rp.gz)
                            : 0);
    n[j] = ok ? 1 : 0;  // a cell the stencil leaves out (tiny grids) is skipped
  }
  int m[14];
#pragma unroll
  for (int j = 0; j < 14; ++j) m[j] = cntb[cell[j]];  // no branch around the loads
#pragma unroll
  for (int j = 0; j < 14; ++j) n[j] = n[j] ? min(m[j], cap) : 0;
  auto hits = [&](const SlotRec &rec, bool own) {
    // compute_dist with sf (moves.c:400-431), reference particle first;
    // in the own cell each pair once, self excluded
    return !(own && rec.id <= me) &&
           dist2_scaled(ax, ay, az, rec.x, rec.y, rec.z, rp.lx, rp.ly, rp.lz, sf) < 1.0;
  };
  bool ov = false;
  for (int j = 0; j < 14 && !ov; ++j) {
    const int c = cell[j];
    const SlotRec r0 = slot[c], r1 = slot[(size_t)(cap > 1 ? 1 : 0) * C + c];
    const int stop = j > 0 ? __hip_atomic_load(&flags[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    if (stop) break;
    ov = (n[j] > 0 && hits(r0, j == 0)) || (n[j] > 1 && hits(r1, j == 0));
    for (int q = 2; q < n[j] && !ov; ++q) ov = hits(slot[(size_t)q * C + c], j == 0);
  }
  if (ov) atomicOr(&flags[r], 1);
}

// A volume move as the host proposes it: its scale factor, whether the
// acceptance rule passes (decided before the scan: it does not depend on
// it), and the replica's record in the new box.
struct VolNode {
  double sf;
  int rule, pad;
  RepDev rec;
};

// One round of volume moves on the device: the replicas whose move passed
// the scan (flags) and the rule take their new record and their spheres
// their scaled positions (moves.c:134-140: coordinates times sf, then
// apply_pbc in the new box).  Block b takes the 256 spheres from blk[b] on,
// all of one replica.  The flags go to the host's copy.
__global__ void __launch_bounds__(256)
k_vol_apply(const int *__restrict__ blk, const int *__restrict__ prep, const VolNode *__restrict__ node,
            const int *__restrict__ flags, RepDev *__restrict__ reps, double *__restrict__ x,
            double *__restrict__ y, double *__restrict__ z, int *__restrict__ host_flags) {
  const int i0 = blk[blockIdx.x], r = prep[i0];
  const VolNode &nd = node[r];
  const double sf = nd.sf;
  const int hit = flags[r], first = nd.rec.poff;
  if (i0 == first && threadIdx.x == 0) host_flags[r] = hit;
  if (!(sf > 0.0) || hit || !nd.rule) return;
  const int i = i0 + (int)threadIdx.x;
  if (i < first + nd.rec.N) {
    x[i] = wrap_once(x[i] * sf, nd.rec.lx);
    y[i] = wrap_once(y[i] * sf, nd.rec.ly);
    z[i] = wrap_once(z[i] * sf, nd.rec.lz);
  }
  if (i0 == first && threadIdx.x == 0) reps[r] = nd.rec;
}

// Several volume moves of small replicas in one launch, a workgroup each.
// Which move follows depends on the one before, so the host lays a replica's
// next moves out as a binary tree (node k: accepted 2 k + 1, else 2 k + 2)
// with its own log, exp and pow, and the kernel walks it.
//
// One scan serves all the moves: the smallest squared distance s of any pair,
// on a search grid filed in LDS whose cells cover the strongest compression
// of the tree.  A move by sf makes an overlap when s sf^2 < 1, and an
// accepted one scales s by sf^2; only where s sf^2 lies within kNear, or
// kNearEdge of the longest edge, of 1 are the pairs tested one by one with
// the reference's arithmetic.  The rounding of the coordinates in up to 3
// accepted moves (2^-53 of the edge each) and of the products moves s by less:
// by 2 (|dx| + |dy| + |dz|) 6 2^-53 < 2.4e-15 of the edge near 1.  Latency-bound, 23 us for the 32 x N = 256
// of the published table (40 us with a scan per move); a sweep's volume moves
// took about 400 us as rounds of transfers and waits.
constexpr int kVolDepth = 4;               // moves per launch at most
constexpr int kVolThreads = 1024;         // threads at most: one per sphere, 256 at least
constexpr int kVolPer = 4;                 // spheres per thread at most
constexpr int kVolSpheres = kVolThreads * kVolPer;
constexpr int kVolAxis = 16;               // search-grid cells per axis at most

// Where one launch of a workgroup a replica is faster than a round of kernels
// on the whole device and a wait for each move (of which some replica of many
// makes more).  us per NpT sweep at density 0.6, one launch / rounds (the waits
// take one of two durations in a process): a single replica of 864 spheres 67 /
// 63 to 75, 2048 75 / 62 to 75, 4000 93 / 62 to 75; four of 864 79 / 106, 2048
// 99 / 96 to 104, 4000 131 / 98 to 105; 16 of 2916 125 / 148, 4000 155 / 157.
constexpr bool moves_in_one_launch(int R, int n_max) { return n_max <= kVolSpheres && n_max <= 1500 + 250L * R; }

constexpr size_t vol_lds_bytes(int N) { return sizeof(double) * 3 * N + sizeof(int) * kVolAxis * kVolAxis * kVolAxis; }
constexpr double kNear = 1e-9, kNearEdge = 1e-14;

struct VolPlan {
  int steps, first;  // moves of this launch and the replica's first node
};

__device__ __forceinline__ int search_cells(double L, double cut) {
  int n = (int)(L / cut);
  n = n < 1 ? 1 : (n > kVolAxis ? kVolAxis : n);
  while (n > 1 && L / n < cut) --n;
  return n;
}

__global__ void __launch_bounds__(kVolThreads)
k_volume_moves(RepDev *__restrict__ reps, const VolPlan *__restrict__ plan,
               const VolNode *__restrict__ nodes, double *__restrict__ gx, double *__restrict__ gy,
               double *__restrict__ gz, int *__restrict__ result) {
  extern __shared__ double vol_lds[];
  __shared__ int tot[kVolThreads / 64];
  __shared__ double low[kVolThreads / 64];
  __shared__ VolNode tree[(1 << kVolDepth) - 1];
  const int r = blockIdx.x, T = blockDim.x, t = threadIdx.x, w = t >> 6;
  const int steps = plan[r].steps;
  if (steps == 0) return;
  // the moves lie in host memory: read once, side by side
  constexpr int words = sizeof(VolNode) / 8;
  static_assert(sizeof(VolNode) % 8 == 0 && words * ((1 << kVolDepth) - 1) <= 256, "one read");
  const int count = (1 << steps) - 1;
  if (t < words * count)
    reinterpret_cast<unsigned long long *>(tree)[t] =
        reinterpret_cast<const unsigned long long *>(nodes + plan[r].first)[t];
  const int N = reps[r].N, poff = reps[r].poff;
  double lx = reps[r].lx, ly = reps[r].ly, lz = reps[r].lz;
  double x[kVolPer], y[kVolPer], z[kVolPer];
#pragma unroll
  for (int u = 0; u < kVolPer; ++u) {
    const int i = min(t + u * T, N - 1);
    x[u] = gx[poff + i];
    y[u] = gy[poff + i];
    z[u] = gz[poff + i];
  }
  double *px = vol_lds, *py = px + N, *pz = py + N;
  int *cnt = reinterpret_cast<int *>(pz + N);  // once filed, the end of each cell
  __syncthreads();
  int nx = 1, ny = 1, nz = 1;
  double ix = 0.0, iy = 0.0, iz = 0.0;  // reciprocal cell sides
  // file the spheres in cells of side at least cut
  auto file = [&](double cut) {
    nx = search_cells(lx, cut);
    ny = search_cells(ly, cut);
    nz = search_cells(lz, cut);
    ix = nx / lx;
    iy = ny / ly;
    iz = nz / lz;
    const int C = nx * ny * nz;
    __syncthreads();  // an earlier filing is no longer read
    for (int c = t; c < C; c += T) cnt[c] = 0;
    __syncthreads();
    int ci[kVolPer], at[kVolPer];
#pragma unroll
    for (int u = 0; u < kVolPer; ++u) {
      if (t + u * T < N) {
        ci[u] = (search_cell(x[u], ix, nx) * ny + search_cell(y[u], iy, ny)) * nz + search_cell(z[u], iz, nz);
        at[u] = atomicAdd(&cnt[ci[u]], 1);
      }
    }
    __syncthreads();
    const int per = (C + T - 1) / T, c0 = min(t * per, C), c1 = min(c0 + per, C);
    int s = 0;
    for (int c = c0; c < c1; ++c) s += cnt[c];
    const int incl = group_inclusive_sum<64>(s);
    if ((t & 63) == 63) tot[w] = incl;
    __syncthreads();
    int run = incl - s;
    for (int k = 0; k < w; ++k) run += tot[k];
    for (int c = c0; c < c1; ++c) {
      run += cnt[c];
      cnt[c] = run;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kVolPer; ++u) {
      if (t + u * T < N) {
        const int p = (ci[u] ? cnt[ci[u] - 1] : 0) + at[u];
        px[p] = x[u];
        py[p] = y[u];
        pz[p] = z[u];
      }
    }
    __syncthreads();
  };
  // the least f(pair) over the pairs of a 27-cell stencil, each once (the
  // spheres after p in filed order), in every thread
  auto least = [&](auto &&f) {
    double m = 1e300;
    for (int p = t; p < N; p += T) {
      const double ax = px[p], ay = py[p], az = pz[p];
      const int cx = search_cell(ax, ix, nx), cy = search_cell(ay, iy, ny), cz = search_cell(az, iz, nz);
      for (int d = 0; d < 27; ++d) {
        const int dx = d / 9 - 1, dy = (d / 3) % 3 - 1, dz = d % 3 - 1;
        if (!stencil_axis_ok(dx, nx) || !stencil_axis_ok(dy, ny) || !stencil_axis_ok(dz, nz)) continue;
        const int c = (wrap_index(cx + dx, nx) * ny + wrap_index(cy + dy, ny)) * nz + wrap_index(cz + dz, nz);
        const int e = cnt[c];
        for (int q = max(c ? cnt[c - 1] : 0, p + 1); q < e; ++q) m = fmin(m, f(ax, ay, az, px[q], py[q], pz[q]));
      }
    }
    for (int o = 32; o > 0; o >>= 1) m = fmin(m, __shfl_xor(m, o, 64));
    __syncthreads();  // low is no longer read
    if ((t & 63) == 0) low[w] = m;
    __syncthreads();
    for (int k = 0; k < T / 64; ++k) m = fmin(m, low[k]);
    return m;
  };
  double sf_min = 1.0;  // along any path: at most kVolDepth compressions in a row
  {
    double least_sf = 1.0;
    for (int k = 0; k < count; ++k) least_sf = fmin(least_sf, tree[k].sf);
    for (int k = 0; k < steps; ++k) sf_min *= least_sf;
  }
  file((1.0 / sf_min) * (1.0 + 1e-6));
  // pairs the grid does not hold are farther apart than 1 / sf_min
  double s = fmin(least([&](double ax, double ay, double az, double bx, double by, double bz) {
                    return dist2(ax, ay, az, bx, by, bz, lx, ly, lz);
                  }),
                  (1.0 + 1e-6) / (sf_min * sf_min));
  int cur = 0, bits = 0, moved = 0;
  for (int k = 0; k < steps; ++k) {
    const double near = fmax(kNear, kNearEdge * fmax(lx, fmax(ly, lz)));
    const double sf = tree[cur].sf, after = s * sf * sf;
    bool hit = false;
    if (sf < 1.0) {  // an expansion makes no overlap
      hit = after < 1.0;
      if (fabs(after - 1.0) < near) {
        file((1.0 / sf) * (1.0 + 1e-6));
        hit = least([&](double ax, double ay, double az, double bx, double by, double bz) {
                return dist2_scaled(ax, ay, az, bx, by, bz, lx, ly, lz, sf);
              }) < 1.0;
      }
    }
    const bool accept = !hit && tree[cur].rule;
    bits |= (hit ? 1 : 0) << k | (accept ? 1 : 0) << (16 + k);
    if (accept) {
      lx = tree[cur].rec.lx;
      ly = tree[cur].rec.ly;
      lz = tree[cur].rec.lz;
#pragma unroll
      for (int u = 0; u < kVolPer; ++u) {
        x[u] = wrap_once(x[u] * sf, lx);
        y[u] = wrap_once(y[u] * sf, ly);
        z[u] = wrap_once(z[u] * sf, lz);
      }
      s = after;
      moved = cur + 1;
    }
    cur = 2 * cur + (accept ? 1 : 2);
  }
  if (moved) {
#pragma unroll
    for (int u = 0; u < kVolPer; ++u) {
      const int i = t + u * T;
      if (i < N) {
        gx[poff + i] = x[u];
        gy[poff + i] = y[u];
        gz[poff + i] = z[u];
      }
    }
    if (t == 0) reps[r] = tree[moved - 1].rec;
  }
  if (t == 0) result[r] = bits;
}

__global__ void k_zero_flags(int *__restrict__ f, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) f[i] = 0;
}

// Uniform in [0, 1] from one Philox output word (rng_get_double's range).
double unit_closed(uint32_t u) { return (double)u / 4294967295.0; }

// Number of volume moves among the N steps of one sweep: Binomial(N, p),
// p = 1/(N+1), by inversion of u in [0, 1).
int volume_steps(int N, uint32_t word) {
  const double u = (double)word * 0x1p-32;
  const double p = 1.0 / (N + 1.0);
  double pk = pow(1.0 - p, N), cdf = pk;
  int k = 0;
  while (u > cdf && k < N) {
    pk *= (double)(N - k) / (double)(k + 1) * p / (1.0 - p);
    ++k;
    cdf += pk;
  }
  return k;
}

void draws(const RepHost &h, unsigned long long sweep, uint32_t round, uint32_t out[4]) {
  philox4x32_10((uint32_t)sweep, (uint32_t)(sweep >> 32), round, kNptTag, (uint32_t)h.p.seed,
                (uint32_t)(h.p.seed >> 32), out);
}

}  // namespace

extern "C" {

int hsmc_gpu_box(const hsmc_gpu_ctx *ctx, int replica, double out[3]) {
  if (!ctx || replica < 0 || replica >= ctx->R || !out) return HSMC_ERR_BAD_ARG;
  out[0] = ctx->reps[replica].p.lx;
  out[1] = ctx->reps[replica].p.ly;
  out[2] = ctx->reps[replica].p.lz;
  return HSMC_OK;
}

}  // extern "C"

namespace {

// First sphere of each 256-sphere block, every block inside one replica, on
// the device (the particle counts of a context do not change).
int sphere_blocks(hsmc_gpu_ctx *ctx, const int **blk, int *n) {
  size_t count = 0;
  for (const RepHost &h : ctx->reps) count += (size_t)(h.p.n_part + 255) / 256;
  const bool had = ctx->scratch_bytes[S_BLK] > 0;
  int *d = (int *)scratch(ctx, S_BLK, sizeof(int) * count);
  if (!d) return HSMC_ERR_NO_MEMORY;
  if (!had) {
    std::vector<int> b;
    b.reserve(count);
    for (const RepHost &h : ctx->reps)
      for (long i = h.poff; i < h.poff + h.p.n_part; i += 256) b.push_back((int)i);
    HSMC_HIP(ctx, hipMemcpyAsync(d, b.data(), sizeof(int) * count, hipMemcpyHostToDevice, ctx->stream));
    HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  }
  *blk = d;
  *n = (int)count;
  return HSMC_OK;
}

// Whether the sweep grid's cells cover the scaled cutoff 1/sf.
bool sweep_grid_covers(const RepHost &h, double sf) {
  const double side = std::min(h.p.lx / h.gx, std::min(h.p.ly / h.gy, h.p.lz / h.gz));
  return side >= (1.0 / sf) * (1.0 + 1e-9);
}

// Enqueue the scan of the replicas with sf[r] > 0 (in device memory) on the
// last sweep's cell list, flags on the device.
int enqueue_scan(hsmc_gpu_ctx *ctx, const double *sf, int *d_flag, const int *blk, int nblk) {
  if (ctx->cells_version != ctx->version) {  // positions changed since the last sweep, or no list in memory
    int st = rebin_last_sweep(ctx);
    if (st) return st;
  }
  const int R = ctx->R;
  hipLaunchKernelGGL(k_zero_flags, dim3((R + 255) / 256), dim3(256), 0, ctx->stream, d_flag, R);
  hipLaunchKernelGGL(k_vol_overlap, dim3((unsigned)nblk), dim3(256), 0, ctx->stream, ctx->d_reps,
                     ctx->d_swp + (ctx->R == 1 ? ctx->swp_last : 0), ctx->R, ctx->d_prep, blk, (int)ctx->Ctot,
                     ctx->d_cnt, ctx->d_slot, ctx->cap, ctx->d_sweep, ctx->d_x, ctx->d_y, ctx->d_z, sf,
                     d_flag);
  HSMC_HIP(ctx, hipGetLastError());
  return HSMC_OK;
}

__global__ void k_copy_flags(const int *__restrict__ f, int n, const unsigned *__restrict__ err,
                             int *__restrict__ host) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) host[i] = f[i];
  if (i == n) host[n] = (int)*err;
}

// A replica's volume move from its present box (moves.c:91-121): the
// proposal and the acceptance rule.
struct Box {
  double lx, ly, lz;
};

VolNode propose(const RepHost &h, const Box &b, unsigned long long sweep, int t, double press, double dv_max,
                Box *next) {
  uint32_t u[4];
  draws(h, sweep, (uint32_t)t + 1u, u);
  const double vol = b.lx * b.ly * b.lz;
  const double log_vol_new = log(vol) + (unit_closed(u[0]) - 0.5) * dv_max;
  const double vnew = exp(log_vol_new);
  VolNode n{};
  n.sf = pow(vnew / vol, 1. / 3.);
  const double boltz = exp(press * (vol - vnew) + (h.p.n_part + 1) * log(vnew / vol));
  n.rule = !(unit_closed(u[1]) >= boltz);
  next->lx = b.lx * n.sf;
  next->ly = b.ly * n.sf;
  next->lz = b.lz * n.sf;
  RepHost hh = h;
  hh.p.lx = next->lx;
  hh.p.ly = next->ly;
  hh.p.lz = next->lz;
  fill_repdev(hh, n.rec);
  return n;
}

void count_move(uint64_t *vc, bool overlap, bool accepted) {
  if (!vc) return;
  vc[0] += 1;
  vc[accepted ? 1 : (overlap ? 2 : 3)] += 1;
}

// After accepted moves: the boxes are in ctx->reps and the records and
// positions on the device already; the layout follows where a grid changed.
int boxes_changed(hsmc_gpu_ctx *ctx) {
  ctx->version++;
  if (layout_keeps(ctx)) return HSMC_OK;
  return layout(ctx);
}

// The volume moves of one sweep, steps[r] of replica r, for replicas that
// fit k_volume_moves.  With *ahead set, the next sweep is enqueued behind the
// last of them where the layout serves every outcome (the resident kernel
// reads boxes and positions on the device), so that it runs while the host
// takes the decisions in and draws the next moves (32 replicas of N = 256: 57
// -> 52 us a sweep); *ahead tells whether it was.
int volume_moves_small(hsmc_gpu_ctx *ctx, unsigned long long sweep, const std::vector<int> &steps, int rounds,
                       const double *press, const double *dv_max, uint64_t *vol_counts, bool *ahead) {
  const bool may = *ahead;
  *ahead = false;
  const int R = ctx->R;
  int n_max = 0;
  for (const RepHost &h : ctx->reps) n_max = std::max(n_max, h.p.n_part);
  const int threads = std::min(kVolThreads, (n_max + 255) / 256 * 256);
  const size_t lds = vol_lds_bytes(n_max);
  // with the kernel's own few KB above 64 KB; always the same value: contexts
  // of other threads launch this kernel too
  if (lds > 60 * 1024)
    HSMC_HIP(ctx, hipFuncSetAttribute((const void *)k_volume_moves, hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)vol_lds_bytes(kVolSpheres)));
  for (int t0 = 0; t0 < rounds; t0 += kVolDepth) {
    // each replica's tree of this launch's moves
    std::vector<VolNode> nodes;
    std::vector<VolPlan> plan(R);
    std::vector<Box> at;
    bool keeps = may && t0 + kVolDepth >= rounds;
    for (int r = 0; r < R; ++r) {
      const RepHost &h = ctx->reps[r];
      const int k = std::max(0, std::min(kVolDepth, steps[r] - t0));
      plan[r] = VolPlan{k, (int)nodes.size()};
      if (k == 0) continue;
      const int n = (1 << k) - 1;
      at.assign(2 * n + 1, Box{h.p.lx, h.p.ly, h.p.lz});
      for (int i = 0, depth = 0; i < n; ++i) {
        if (i == (2 << depth) - 1) ++depth;
        nodes.push_back(propose(h, at[i], sweep, t0 + depth, press[r], dv_max[r], &at[2 * i + 1]));
        keeps = keeps && box_fits_layout(ctx, h, nodes.back().rec);
        at[2 * i + 2] = at[i];
      }
    }
    const size_t o_node = (sizeof(VolPlan) * R + 15) & ~(size_t)15;
    const size_t o_res = o_node + sizeof(VolNode) * nodes.size();
    unsigned char *host = (unsigned char *)pinned(ctx, P_MOVES, o_res + sizeof(int) * R);
    if (!host) return HSMC_ERR_NO_MEMORY;
    memcpy(host, plan.data(), sizeof(VolPlan) * R);
    memcpy(host + o_node, nodes.data(), sizeof(VolNode) * nodes.size());
    const int *res = (const int *)(host + o_res);
    hipLaunchKernelGGL(k_volume_moves, dim3((unsigned)R), dim3((unsigned)threads), lds, ctx->stream, ctx->d_reps,
                       (const VolPlan *)host, (const VolNode *)(host + o_node), ctx->d_x, ctx->d_y, ctx->d_z,
                       (int *)(host + o_res));
    HSMC_HIP(ctx, hipGetLastError());
    // a sweep that cannot be enqueued (an error of the last one, say) is
    // reported once the moves above are taken in: they are done on the device
    int sweep_status = HSMC_OK;
    if (keeps) {
      HSMC_HIP(ctx, hipEventRecord(ctx->ev0, ctx->stream));
      sweep_status = run_sweeps(ctx, 1);
      *ahead = sweep_status == HSMC_OK;
      HSMC_HIP(ctx, hipEventSynchronize(ctx->ev0));
    } else {
      HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    }
    bool any = false;
    for (int r = 0; r < R; ++r) {
      int cur = 0;
      for (int k = 0; k < plan[r].steps; ++k) {
        const bool acc = (res[r] >> (16 + k)) & 1, ov = (res[r] >> k) & 1;
        count_move(vol_counts ? vol_counts + 4 * (size_t)r : nullptr, ov, acc);
        if (acc) {
          const RepDev &rec = nodes[plan[r].first + cur].rec;
          hsmc_gpu_replica &p = ctx->reps[r].p;
          p.lx = rec.lx;
          p.ly = rec.ly;
          p.lz = rec.lz;
          any = true;
        }
        cur = 2 * cur + (acc ? 1 : 2);
      }
    }
    if (any) {
      int st = boxes_changed(ctx);
      if (st) return st;
    }
    if (sweep_status) return sweep_status;
  }
  return HSMC_OK;
}

// The same round by round for any replicas: round t holds the t-th move of
// every replica that makes more than t, scanned on the last sweep's cells.
int volume_moves_rounds(hsmc_gpu_ctx *ctx, unsigned long long sweep, const std::vector<int> &steps, int rounds,
                        const double *press, const double *dv_max, uint64_t *vol_counts) {
  const int R = ctx->R;
  const int *blk = nullptr;
  int nblk = 0, st = sphere_blocks(ctx, &blk, &nblk);
  if (st) return st;
  int *d_flag = (int *)scratch(ctx, S_FLAG, sizeof(int) * R);
  if (!d_flag) return HSMC_ERR_NO_MEMORY;
  const size_t o_sf = sizeof(VolNode) * R, o_res = o_sf + sizeof(double) * R;
  unsigned char *host = (unsigned char *)pinned(ctx, P_MOVES, o_res + sizeof(int) * R);
  if (!host) return HSMC_ERR_NO_MEMORY;
  VolNode *node = (VolNode *)host;
  double *sf = (double *)(host + o_sf);
  const int *flag = (const int *)(host + o_res);
  // the blocks of a round read their replica's move from device memory
  unsigned char *dev = (unsigned char *)scratch(ctx, S_MOVE, o_res);
  if (!dev) return HSMC_ERR_NO_MEMORY;
  std::vector<uint8_t> decided(R);  // overlap found by the single scan
  for (int t = 0; t < rounds; ++t) {
    bool scan = false;
    for (int r = 0; r < R; ++r) {
      const RepHost &h = ctx->reps[r];
      decided[r] = 0;
      sf[r] = 0.0;
      Box next;
      if (steps[r] <= t) {
        node[r] = VolNode{};
        fill_repdev(h, node[r].rec);
        continue;
      }
      node[r] = propose(h, Box{h.p.lx, h.p.ly, h.p.lz}, sweep, t, press[r], dv_max[r], &next);
      // an expansion cannot create an overlap in a configuration that has none
      if (!(node[r].sf < 1.0)) continue;
      if (sweep_grid_covers(h, node[r].sf)) {
        sf[r] = node[r].sf;
        scan = true;
      } else {
        uint8_t ok = 1;
        st = hsmc_gpu_any_overlap_scaled(ctx, r, &node[r].sf, 1, &ok);
        if (st) return st;
        decided[r] = !ok;
        if (decided[r]) node[r].rule = 0;
      }
    }
    HSMC_HIP(ctx, hipMemcpyAsync(dev, host, o_res, hipMemcpyHostToDevice, ctx->stream));
    if (scan) {
      st = enqueue_scan(ctx, (const double *)(dev + o_sf), d_flag, blk, nblk);
      if (st) return st;
    } else {
      hipLaunchKernelGGL(k_zero_flags, dim3((R + 255) / 256), dim3(256), 0, ctx->stream, d_flag, R);
    }
    hipLaunchKernelGGL(k_vol_apply, dim3((unsigned)nblk), dim3(256), 0, ctx->stream, blk, ctx->d_prep,
                       (const VolNode *)dev, d_flag, ctx->d_reps, ctx->d_x, ctx->d_y, ctx->d_z, (int *)(host + o_res));
    HSMC_HIP(ctx, hipGetLastError());
    HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    bool any = false;
    for (int r = 0; r < R; ++r) {
      if (steps[r] <= t) continue;
      const bool ov = decided[r] || flag[r], acc = !ov && node[r].rule;
      count_move(vol_counts ? vol_counts + 4 * (size_t)r : nullptr, ov, acc);
      if (!acc) continue;
      hsmc_gpu_replica &p = ctx->reps[r].p;
      p.lx = node[r].rec.lx;
      p.ly = node[r].rec.ly;
      p.lz = node[r].rec.lz;
      any = true;
    }
    if (any) {
      st = boxes_changed(ctx);
      if (st) return st;
    }
  }
  return HSMC_OK;
}

}  // namespace

extern "C" {

int hsmc_gpu_any_overlap_scaled_batch(hsmc_gpu_ctx *ctx, const double *sf, uint8_t *no_overlap) {
  if (!ctx || !sf || !no_overlap) return HSMC_ERR_BAD_ARG;
  const int R = ctx->R;
  int *d_flag = (int *)scratch(ctx, S_FLAG, sizeof(int) * R);
  if (!d_flag) return HSMC_ERR_NO_MEMORY;
  // replicas whose sweep-grid cells cover the scaled cutoff 1/sf are scanned
  // together on the sweep grid; the others one by one
  std::vector<double> on_grid(R, 0.0);
  bool any = false;
  for (int r = 0; r < R; ++r) {
    no_overlap[r] = 1;
    if (!(sf[r] > 0.0)) continue;
    if (sweep_grid_covers(ctx->reps[r], sf[r])) {
      on_grid[r] = sf[r];
      any = true;
    } else {
      int st = hsmc_gpu_any_overlap_scaled(ctx, r, &sf[r], 1, &no_overlap[r]);
      if (st) return st;
    }
  }
  if (!any) return HSMC_OK;
  const int *blk = nullptr;
  int nblk = 0, st = sphere_blocks(ctx, &blk, &nblk);
  if (st) return st;
  unsigned char *host = (unsigned char *)pinned(ctx, P_MOVES, sizeof(double) * R + sizeof(int) * (R + 1));
  if (!host) return HSMC_ERR_NO_MEMORY;
  memcpy(host, on_grid.data(), sizeof(double) * R);
  int *flag = (int *)(host + sizeof(double) * R);
  double *d_sf = (double *)scratch(ctx, S_MOVE, sizeof(double) * R);
  if (!d_sf) return HSMC_ERR_NO_MEMORY;
  HSMC_HIP(ctx, hipMemcpyAsync(d_sf, host, sizeof(double) * R, hipMemcpyHostToDevice, ctx->stream));
  st = enqueue_scan(ctx, d_sf, d_flag, blk, nblk);
  if (st) return st;
  hipLaunchKernelGGL(k_copy_flags, dim3((unsigned)(R / 256 + 1)), dim3(256), 0, ctx->stream, d_flag, R, ctx->d_err, flag);
  HSMC_HIP(ctx, hipGetLastError());
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  for (int r = 0; r < R; ++r)
    if (on_grid[r] > 0.0) no_overlap[r] = flag[r] ? 0 : 1;
  return flag[R] ? check_device_errors(ctx) : HSMC_OK;
}

int hsmc_gpu_npt_sweeps(hsmc_gpu_ctx *ctx, int n_sweeps, const double *press,
                        const double *dv_max, uint64_t *vol_counts) {
  if (!ctx || n_sweeps < 0 || !press || !dv_max) return HSMC_ERR_BAD_ARG;
  const int R = ctx->R;
  for (int r = 0; r < R; ++r)
    if (!(press[r] >= 0.0) || !(dv_max[r] > 0.0) || !std::isfinite(press[r])) return HSMC_ERR_BAD_ARG;
  if (n_sweeps == 0) return HSMC_OK;
  const unsigned long long sweep0 = ctx->sweep_now;
  int n_max = 0;
  for (const RepHost &h : ctx->reps) n_max = std::max(n_max, (int)h.p.n_part);
  const bool small = moves_in_one_launch(R, n_max);
  std::vector<int> steps(R);
  ResidentShape shape;
  bool ahead = false;  // the sweep was enqueued behind the last one's volume moves
  for (int sw = 0; sw < n_sweeps; ++sw) {
    int st = ahead ? HSMC_OK : run_sweeps(ctx, 1);
    if (st) return st;
    const unsigned long long s = sweep0 + (unsigned long long)sw;  // the sweep just done
    int rounds = 0;
    for (int r = 0; r < R; ++r) {
      uint32_t u[4];
      draws(ctx->reps[r], s, 0u, u);
      steps[r] = volume_steps(ctx->reps[r].p.n_part, u[0]);
      rounds = std::max(rounds, steps[r]);
    }
    ahead = small && sw + 1 < n_sweeps && !ctx->tune_set && resident_shape(ctx, &shape);
    if (rounds == 0) ahead = false;
    st = small ? volume_moves_small(ctx, s, steps, rounds, press, dv_max, vol_counts, &ahead)
               : volume_moves_rounds(ctx, s, steps, rounds, press, dv_max, vol_counts);
    if (st) return st;
  }
  return check_device_errors(ctx);
}

}  // extern "C"
