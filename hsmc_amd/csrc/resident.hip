// resident.hip -- checkerboard sweeps of small systems in one launch.
//
// A sweep of a few hundred spheres is a few dozen active cells per sublattice
// phase: launched phase by phase it is nothing but latency (a kernel boundary
// and three rounds of dependent loads per phase).  Here one workgroup per
// replica keeps the whole system in LDS and runs any number of sweeps, with a
// workgroup barrier in place of each kernel boundary.  The moves, draws,
// decisions and their order are those of the launched kernels (sweep.hip):
// the same trajectory bit for bit, the same counters, the same errors.
//
// Per sweep, one thread per sphere files it into the shifted grid, ranks it
// by id among its cell's occupants, and prepares one attempt: the cell's
// attempt t belongs to its occupant of rank t, so the N attempts of a sweep
// are drawn by N lanes at once (the launched phase kernel draws them in 32
// lanes per cell, most of them idle).  A prepared trial holds as long as its
// sphere has not moved since, and only an earlier attempt of the same cell
// can have moved it; that attempt's draw is made again from the new position.
//
// Per phase, LPC lanes take an active cell: they gather the ids of the 27
// cells' spheres into a list and its first RC * LPC positions into registers,
// then make the cell's attempts one after the other, each broadcast from the
// lane that holds it.  What bounds it is the instructions of these steps on
// the four SIMDs of one compute unit and their latency: of 18.9 us per sweep
// at N = 256, filing and drawing take 1.5, gathering 5.7 and the attempts the
// rest (34 us with a launch per phase).
#include <stdio.h>

#include <algorithm>

#include "ctx.h"
#include "device_common.h"
#include "sweep_draws.h"

using namespace hsmc;

namespace {

constexpr int kDrawTable = 64;  // sweeps whose shift and order are drawn together
constexpr int kMaxPer = 4;      // spheres per thread at most
constexpr unsigned kStays = 0x8000u;
constexpr size_t kMaxLds = 160 * 1024;

// Inclusive sum over groups of LPC (16 or 32) lanes.  A group of 16 is a DPP
// row: shifts by 1, 2, 4 and 8 within it, a shifted-in lane reading 0.
template <int LPC>
__device__ __forceinline__ int lane_sum(int v) {
  if constexpr (LPC == 32) return group_inclusive_sum<32>(v);
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
  return v;
}

// LDS of one replica: positions and prepared trials (doubles), the table of
// shifts and orders, occupants by cell and rank, the attempts' draws, counts
// and active cells' coordinates (32-bit), attempt words and the groups' lists
// (16-bit).
struct Layout {
  int trial, table, occ, draw, cnt, act, att, list, bytes;
};

__host__ __device__ inline Layout resident_layout(int N, int C, int cap, int groups, int lcap) {
  Layout l;
  int o = 24 * N;
  l.trial = o;
  o += 24 * N;
  l.table = o;
  o += kDrawTable * (int)sizeof(SweepDev);
  l.occ = o;
  o += 2 * cap * C;
  l.draw = o;
  o += 12 * N;
  l.cnt = o;
  o += 4 * C;
  l.act = o;
  o += 4 * ((C + 7) / 8);
  l.att = o;
  o += 2 * N;
  l.list = o;
  o += 2 * lcap * groups;
  l.bytes = (o + 15) & ~15;
  return l;
}

template <int CAP, int LPC, int RC>
__global__ void __launch_bounds__(1024)
k_sweeps_resident(const RepDev *__restrict__ reps, int lcap, double *__restrict__ x,
                  double *__restrict__ y, double *__restrict__ z, unsigned long long base,
                  unsigned long long *__restrict__ sweep_counter, int n_sweeps,
                  unsigned int *__restrict__ cacc, unsigned int *__restrict__ cleft,
                  unsigned int *__restrict__ err, unsigned int *__restrict__ host_err) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const RepDev rp = reps[blockIdx.x];
  const int T = blockDim.x, tid = threadIdx.x, groups = T / LPC;
  const int N = rp.N, C = rp.gx * rp.gy * rp.gz, A = C / 8;
  const Layout l = resident_layout(N, C, CAP, groups, lcap);
  double *px = reinterpret_cast<double *>(lds), *py = px + N, *pz = py + N;
  double *tx = reinterpret_cast<double *>(lds + l.trial), *ty = tx + N, *tz = ty + N;
  SweepDev *table = reinterpret_cast<SweepDev *>(lds + l.table);
  int *cnt = reinterpret_cast<int *>(lds + l.cnt);
  unsigned *act = reinterpret_cast<unsigned *>(lds + l.act);
  uint16_t *occ = reinterpret_cast<uint16_t *>(lds + l.occ);
  uint16_t *att = reinterpret_cast<uint16_t *>(lds + l.att);
  uint32_t *d1 = reinterpret_cast<uint32_t *>(lds + l.draw), *d2 = d1 + N, *d3 = d2 + N;
  const int lane = tid & (LPC - 1), grp = tid / LPC;
  uint16_t *list = reinterpret_cast<uint16_t *>(lds + l.list) + grp * lcap;
  const unsigned long long gmask = ((1ull << LPC) - 1) << (tid & 63 & ~(LPC - 1));

  for (int i = tid; i < N; i += T) {
    px[i] = x[rp.poff + i];
    py[i] = y[rp.poff + i];
    pz[i] = z[rp.poff + i];
  }
  for (int c = tid; c < C; c += T) cnt[c] = 0;
  {
    const int hz = rp.gz >> 1, hy = rp.gy >> 1;  // even cell coordinates of each active cell
    for (int a = tid; a < A; a += T)
      act[a] = (unsigned)(2 * (a / (hz * hy))) | (unsigned)(2 * ((a / hz) % hy)) << 10 |
               (unsigned)(2 * (a % hz)) << 20;
  }
  __syncthreads();
  const unsigned act0 = act[grp < A ? grp : 0];
  // the stencil cells of this lane (distinct cells only on 2-cell axes)
  constexpr int JPL = (27 + LPC - 1) / LPC;
  int jx[JPL], jy[JPL], jz[JPL];
  bool jok[JPL];
#pragma unroll
  for (int q = 0; q < JPL; ++q) {
    const int j = lane + q * LPC;
    jx[q] = j / 9 - 1;
    jy[q] = (j / 3) % 3 - 1;
    jz[q] = j % 3 - 1;
    jok[q] = j < 27 && stencil_axis_ok(jx[q], rp.gx) && stencil_axis_ok(jy[q], rp.gy) &&
             stencil_axis_ok(jz[q], rp.gz);
  }
  unsigned bad = 0;  // sticky error bits
  unsigned n_acc = 0, n_left = 0;
  // the cell a position lies in, -1 left of the grid
  auto in_cell = [&](double px_, double py_, double pz_, const SweepDev &sw) {
    const int cx = shifted_cell(px_, sw.shx, rp.lx, rp.ix, rp.gx), cy = shifted_cell(py_, sw.shy, rp.ly, rp.iy, rp.gy),
              cz = shifted_cell(pz_, sw.shz, rp.lz, rp.iz, rp.gz);
    return (cx | cy | cz) < 0 ? -1 : (cx * rp.gy + cy) * rp.gz + cz;
  };
  auto file_cell = [&](double px_, double py_, double pz_, const SweepDev &sw) {
    return (filed_cell(px_, sw.shx, rp.lx, rp.ix, rp.gx) * rp.gy +
            filed_cell(py_, sw.shy, rp.ly, rp.iy, rp.gy)) * rp.gz +
           filed_cell(pz_, sw.shz, rp.lz, rp.iz, rp.gz);
  };
  // an attempt's draw applied to its sphere at (bx, by, bz)
  auto trial = [&](uint32_t w1, uint32_t w2, uint32_t w3, double bx, double by, double bz,
                   double &nx, double &ny, double &nz) {
    nx = wrap_once(bx + (u32_unit_closed(w1) - 0.5) * rp.dr_max, rp.lx);
    ny = wrap_once(by + (u32_unit_closed(w2) - 0.5) * rp.dr_max, rp.ly);
    nz = wrap_once(bz + (u32_unit_closed(w3) - 0.5) * rp.dr_max, rp.lz);
  };
  for (int s = 0; s < n_sweeps; ++s) {
    const unsigned long long sweep = base + (unsigned long long)s;
    if (s % kDrawTable == 0) {
      __syncthreads();  // the last sweep's entry is no longer read
      if (tid < kDrawTable && s + tid < n_sweeps) {
        SweepDev d;
        sweep_shift(rp, sweep + tid, d.shx, d.shy, d.shz);
        d.order = sweep_order(rp, sweep + tid);
        d.pad = 0u;
        table[tid] = d;
      }
    }
    __syncthreads();
    const SweepDev sw = table[s % kDrawTable];
    // file
    int ci[kMaxPer], rank[kMaxPer];
#pragma unroll
    for (int u = 0; u < kMaxPer; ++u) {
      const int i = tid + u * T;
      ci[u] = -1;
      if (i < N) {
        const int c = file_cell(px[i], py[i], pz[i], sw);
        const int sl = atomicAdd(&cnt[c], 1);
        if (sl < CAP) {
          occ[c * CAP + sl] = (uint16_t)i;
          ci[u] = c;
        } else {
          bad |= kErrOverflow;
        }
      }
    }
    __syncthreads();
    // rank by id
#pragma unroll
    for (int u = 0; u < kMaxPer; ++u) {
      const int i = tid + u * T;
      rank[u] = 0;
      if (ci[u] >= 0) {
        const int n = min(cnt[ci[u]], CAP);
        for (int q = 0; q < n; ++q) rank[u] += (int)occ[ci[u] * CAP + q] < i ? 1 : 0;
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kMaxPer; ++u)
      if (ci[u] >= 0) occ[ci[u] * CAP + rank[u]] = (uint16_t)(tid + u * T);
    __syncthreads();
    // prepare attempt `rank` of the sphere's cell: its word is the id of the
    // sphere it moves and whether the trial stays in the cell
#pragma unroll
    for (int u = 0; u < kMaxPer; ++u) {
      const int i = tid + u * T;
      if (ci[u] >= 0) {
        const int c = ci[u], n = min(cnt[c], CAP);
        uint32_t w[4];
        philox4x32_10((uint32_t)c, (uint32_t)rank[u], (uint32_t)sweep, (uint32_t)(sweep >> 32), rp.k0,
                      rp.k1, w);
        const uint32_t k = occupant_pick(w[0], (uint32_t)n, (uint32_t)c, (uint32_t)rank[u], sweep, rp.k0,
                                         rp.k1);
        const int m = occ[c * CAP + k];
        double nx, ny, nz;
        trial(w[1], w[2], w[3], px[m], py[m], pz[m], nx, ny, nz);
        d1[i] = w[1];
        d2[i] = w[2];
        d3[i] = w[3];
        tx[i] = nx;
        ty[i] = ny;
        tz[i] = nz;
        att[i] = (uint16_t)((unsigned)m | (in_cell(nx, ny, nz, sw) == c ? kStays : 0u));
      }
    }
    __syncthreads();
    for (int ph = 0; ph < 8; ++ph) {
      const unsigned colour = (sw.order >> (4 * ph)) & 0xFu;
      for (int a0 = 0; a0 < A; a0 += groups) {
        const int a = a0 + grp;
        const unsigned ac = a0 == 0 ? act0 : act[a < A ? a : 0];
        const int cx = (int)(ac & 1023u) + (int)(colour & 1u), cy = (int)((ac >> 10) & 1023u) + (int)((colour >> 1) & 1u),
                  cz = (int)(ac >> 20) + (int)((colour >> 2) & 1u);
        const int c0 = (cx * rp.gy + cy) * rp.gz + cz;
        const int nc = a < A ? min(cnt[c0], CAP) : 0;
        // counts of the 27 cells, JPL to a lane
        int nb[JPL], nn[JPL], mine = 0;
        uint2 ids[JPL];
#pragma unroll
        for (int q = 0; q < JPL; ++q) {
          nb[q] = jok[q] ? (wrap_index(cx + jx[q], rp.gx) * rp.gy + wrap_index(cy + jy[q], rp.gy)) * rp.gz +
                               wrap_index(cz + jz[q], rp.gz)
                         : 0;
          nn[q] = cnt[nb[q]];
          ids[q] = *reinterpret_cast<const uint2 *>(&occ[nb[q] * CAP]);  // the first 4, beside the count
        }
#pragma unroll
        for (int q = 0; q < JPL; ++q) {
          nn[q] = jok[q] ? min(nn[q], CAP) : 0;
          mine += nn[q];
        }
        if (nc == 0) continue;  // the group
        // lane t < nc holds attempt t: its occupant and prepared trial
        const int it = occ[c0 * CAP + (lane < nc ? lane : 0)];
        unsigned word = att[it];
        const int incl = lane_sum<LPC>(mine);
        const int total = __shfl(incl, LPC - 1, LPC);
        if (total > lcap) {  // above the host's packing bound: overlapping spheres
          bad |= kErrListFull;
          continue;
        }
        int o = incl - mine;
#pragma unroll
        for (int q = 0; q < JPL; ++q) {
          if (nn[q] > 0) list[o] = (uint16_t)ids[q].x;
          if (nn[q] > 1) list[o + 1] = (uint16_t)(ids[q].x >> 16);
          if (nn[q] > 2) list[o + 2] = (uint16_t)ids[q].y;
          if (nn[q] > 3) list[o + 3] = (uint16_t)(ids[q].y >> 16);
          for (int e = 4; e < nn[q]; ++e) list[o + e] = occ[nb[q] * CAP + e];
          o += nn[q];
        }
        double nx = tx[it], ny = ty[it], nz = tz[it];
        wave_lds_sync();
        // the list's first RC * LPC spheres in registers; a lane past its end
        // holds a sphere no trial can meet
        int id[RC];
        double qx[RC], qy[RC], qz[RC];
#pragma unroll
        for (int j = 0; j < RC; ++j) {
          const int e = lane + j * LPC;
          id[j] = list[e < total ? e : 0];
          qx[j] = px[id[j]];
          qy[j] = py[id[j]];
          qz[j] = pz[id[j]];
          if (e >= total) id[j] = -1, qx[j] = 1e300;
        }
        for (int t = 0; t < nc; ++t) {
          const unsigned wt = (unsigned)__shfl((int)word, t, LPC);
          const double ax = __shfl(nx, t, LPC), ay = __shfl(ny, t, LPC), az = __shfl(nz, t, LPC);
          if (!(wt & kStays)) {
            ++n_left;
            continue;
          }
          const int m = (int)(wt & ~kStays);
          bool ov = false;
#pragma unroll
          for (int j = 0; j < RC; ++j) {
            const double d2 = dist2(ax, ay, az, qx[j], qy[j], qz[j], rp.lx, rp.ly, rp.lz);
            ov |= (d2 < 1.0) & (id[j] != m);
          }
          for (int e = lane + RC * LPC; e < total; e += LPC) {
            const int k = list[e];
            const double d2 = dist2(ax, ay, az, px[k], py[k], pz[k], rp.lx, rp.ly, rp.lz);
            ov |= (d2 < 1.0) & (k != m);
          }
          if ((__ballot(ov) & gmask) == 0ull) {
            if (lane == t) {
              px[m] = ax;
              py[m] = ay;
              pz[m] = az;
            }
            ++n_acc;
#pragma unroll
            for (int j = 0; j < RC; ++j)
              if (id[j] == m) qx[j] = ax, qy[j] = ay, qz[j] = az;
            if (lane > t && lane < nc && (int)(word & ~kStays) == m) {
              // the sphere's next attempt starts from its new position (the
              // draw is read here: kept in registers, or drawn again, it
              // would be made for every attempt)
              trial(d1[it], d2[it], d3[it], ax, ay, az, nx, ny, nz);
              word = (unsigned)m | (in_cell(nx, ny, nz, sw) == c0 ? kStays : 0u);
            }
          }
          wave_lds_sync();
        }
      }
      __syncthreads();
    }
    for (int c = tid; c < C; c += T) cnt[c] = 0;
  }
  __syncthreads();
  for (int i = tid; i < N; i += T) {
    x[rp.poff + i] = px[i];
    y[rp.poff + i] = py[i];
    z[rp.poff + i] = pz[i];
  }
  if (bad) {  // for the device's readers, and the host's copy at once
    atomicOr(err, bad);
    *host_err = bad;
  }
  // the first sweep's number came by value, so the counter is only written
  if (blockIdx.x == 0 && tid == 0) *sweep_counter = base + (unsigned long long)n_sweeps;
  if (lane == 0 && grp < A) {
    if (n_acc) atomicAdd(&cacc[rp.aoff + grp], n_acc);
    if (n_left) atomicAdd(&cleft[rp.aoff + grp], n_left);
  }
}

using ResidentFn = void (*)(const RepDev *, int, double *, double *, double *, unsigned long long,
                            unsigned long long *, int, unsigned int *, unsigned int *, unsigned int *,
                            unsigned int *);

// Lanes per active cell: 32 while a phase's cells fit the workgroup's 32 such
// groups (us per sweep at N = 108 and 256, 8 and 27 cells a phase: 17.0 and
// 18.9, against 19.6 and 19.9 with 16), else 16 (N = 500, 864 and 1372, 64,
// 125 and 216 cells: 25.3, 43.4 and 67.5, against 32.2, 55.0 and 83.9).
constexpr int kWide = 32, kNarrow = 16;

ResidentFn resident_fn(int cap, int lpc) {
  if (lpc == kWide) return cap == 8 ? k_sweeps_resident<8, kWide, 2> : k_sweeps_resident<16, kWide, 2>;
  return cap == 8 ? k_sweeps_resident<8, kNarrow, 3> : k_sweeps_resident<16, kNarrow, 3>;
}

}  // namespace

namespace hsmc {

// Shape of the resident kernel for the context's replicas; false where they
// do not fit in LDS or launched sweeps are faster.  Measured per sweep: the
// resident kernel takes about 12 + 0.11 A + 0.0225 N us with A active cells a
// phase and N spheres in its largest replica, for as many replicas as there are
// compute units; the launched phases (in their default shape) take 35 us for
// one replica, 42 for several, and 0.0029 us for each active cell of all (A =
// 64 and N = 500 at density 0.85: 26 us against 34 for one replica, 44 for 32,
// 89 for 256; 125 and 864: 43 against 34, 47, 135; 125 and 1372: 57 against 41,
// 58, 176).
bool resident_shape(const hsmc_gpu_ctx *ctx, ResidentShape *shape) {
  long n_max = 0, a_max = 0;
  for (int r = 0; r < ctx->R; ++r) {
    const RepHost &h = ctx->reps[r];
    n_max = std::max(n_max, (long)h.p.n_part);
    a_max = std::max(a_max, (long)h.gx * h.gy * h.gz / 8);
    if (h.gx > 1022 || h.gy > 1022 || h.gz > 1022) return false;
  }
  if (n_max > 1024 * kMaxPer || a_max > 1024) return false;
  const double turns = (double)((ctx->R + ctx->n_cu - 1) / ctx->n_cu);
  if (turns * (12.0 + 0.11 * a_max + 0.0225 * n_max) > (ctx->R == 1 ? 35.0 : 42.0) + 0.0029 * (double)ctx->Atot)
    return false;
  shape->lpc = a_max <= 1024 / kWide ? kWide : kNarrow;
  shape->threads = 256;
  while (shape->threads < 1024 &&
         (shape->threads * kMaxPer < n_max || shape->threads / shape->lpc < a_max))
    shape->threads *= 2;
  shape->bytes = 0;
  for (int r = 0; r < ctx->R; ++r) {
    const RepHost &h = ctx->reps[r];
    const Layout l = resident_layout(h.p.n_part, h.gx * h.gy * h.gz, ctx->cap, shape->threads / shape->lpc, ctx->lcap);
    shape->bytes = std::max(shape->bytes, (size_t)l.bytes);
  }
  return shape->bytes <= kMaxLds;
}

int launch_resident(hsmc_gpu_ctx *ctx, const ResidentShape &shape, unsigned long long base, int n) {
  ResidentFn fn = resident_fn(ctx->cap, shape.lpc);
  // always the same value: contexts of other threads launch this kernel too
  if (shape.bytes > 64 * 1024)
    HSMC_HIP(ctx, hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds));
  hipLaunchKernelGGL(fn, dim3((unsigned)ctx->R), dim3((unsigned)shape.threads), shape.bytes, ctx->stream, ctx->d_reps,
                     ctx->lcap, ctx->d_x, ctx->d_y, ctx->d_z, base, ctx->d_sweep, n, ctx->d_cacc, ctx->d_cleft,
                     ctx->d_err, (unsigned int *)ctx->h_err);
  HSMC_HIP(ctx, hipGetLastError());
  return HSMC_OK;
}

}  // namespace hsmc
