// bricks.hip -- sublattice phases of many replicas or large ones, a brick of
// cells at a time.
//
// The same phase as sweep.hip's k_phase (same attempts, draws, arithmetic and
// cell lists), for contexts with active cells enough to fill the device.
// There a group of 32 lanes for each cell spends its time on what every cell
// needs and few lanes do: 27 counts, a prefix sum, draws for one or two
// attempts, 20 scattered records that 26 other cells read again.  Here a
// workgroup takes a brick of up to 128 active cells: their neighbourhood (11
// cells for each active one in place of 27) is read once, in runs along z,
// into a list in LDS; a lane draws an attempt; 4 lanes test an active cell's
// attempts one after another.
//
// 256 replicas of N = 4000 at density 0.6: 30 us a phase, 65 us cell by cell
// (a sweep 256 and 525 us); N = 10^6 at density 0.9: a sweep 270 and 383 us.
// Bounded by instruction issue (about 1100 vector instructions a wave: a
// third the counts and list, a third the pair tests) and by what a workgroup
// waits for on its way (10 us alone on the device), which 5 workgroups a
// compute unit overlap: lists and registers are held to that (1280 spheres
// and 4 workgroups: 304 us for the 253; 80 registers and 6, spilling: 288).
// The loops are kept rolled: a workgroup runs through its code once or
// twice, so its size is what the instruction cache misses.
//
// LDS holds each sphere's position in the brick's own frame in FP32, one
// 16-byte read a test and no minimum image.  A squared distance outside
// 1 -+ kBand decides; one inside, or any where a sphere lies (or a step may
// lead) outside the box, is decided by the reference's FP64 arithmetic on the
// FP64 positions, so every decision is the FP64 one: coordinates in the
// frame stay below 32 diameters, so each is within 9.6e-7 of its value, a
// difference within 2e-6 (with its rounding), and the squared distance
// within 2 (|dx| + |dy| + |dz|) 2e-6 < 7.2e-6 of its own near 1.
#include <algorithm>
#include <cmath>
#include <vector>

#include "ctx.h"
#include "device_common.h"
#include "sweep_draws.h"

using namespace hsmc;

namespace {

constexpr int kThreads = 256;
constexpr int kActive = 128;    // active cells of a brick, at most
constexpr int kPer = 5;         // cells staged by a thread
constexpr int kRegion = kPer * kThreads;  // cells of a neighbourhood, at most
constexpr int kSide = 2 * 16 + 1;  // and along an axis
constexpr int kSpheres = 896;  // spheres of a neighbourhood that fit
constexpr int kAttempts = 160;  // attempts (and occupants) of a brick that fit
constexpr int kRecs = 3;         // records a thread has in flight
constexpr int kRead = 4;         // entries a lane has in flight
constexpr float kBand = 2e-5f;

static_assert(27 * 16 <= kSpheres && 16 <= kAttempts, "one cell's stencil always fits");
static_assert(kRegion <= 2048, "a region cell's index has 11 bits");

// The value of v, uniform, as if computed here: what is derived from it is not
// moved ahead of the loops (the draws' 20 round keys and the divisors of the
// rare path would take registers throughout the kernel).
__device__ __forceinline__ int here(int v) {
  asm volatile("" : "+s"(v));
  return v;
}

// Whether v lies outside [0, L] by more than 2^-20 of L (a step wider than two
// boxes leads there), by the high words: a negative number's is the larger.
__device__ __forceinline__ bool outside(double v, double L) {
  return (unsigned)__double2hiint(v) > (unsigned)__double2hiint(L);
}

template <int CAP>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(5)))
k_brick_phase(const unsigned long long *__restrict__ sweep_base, const SweepDev *__restrict__ swp,
              const RepDev *__restrict__ reps, const Brick *__restrict__ bricks, int nb, int one,
              int phase, int k, int lcap, double *__restrict__ x, double *__restrict__ y,
              double *__restrict__ z, const int *__restrict__ cnt, int C, SlotRec *__restrict__ slot_all,
              unsigned int *__restrict__ cacc, unsigned int *__restrict__ cleft,
              unsigned int *__restrict__ err) {
  __shared__ float4 list[kSpheres];              // x, y, z in the frame; id (active cells) or record index
  __shared__ double pos[3][kAttempts];           // the occupants, slot by slot of each active cell
  __shared__ uint32_t draw[3][kAttempts];        // each attempt's displacement, drawn
  __shared__ unsigned char slot_of[kAttempts];   // and its occupant's slot
  __shared__ unsigned short start[kRegion + 1];  // a region cell's first list entry
  __shared__ unsigned short first_att[kActive];  // an active cell's first attempt
  __shared__ unsigned char att_cell[kAttempts];  // an attempt's active cell
  __shared__ unsigned char order[kActive];
  __shared__ int act_at[kActive];                // an active cell's place along x, y, z
  __shared__ double centre[3][kSide];            // the region's cell centres along each axis
  __shared__ int cell_at[3][kSide];              // and what a cell's index takes from each axis
  __shared__ int chunk_sum[kPer * 4], bin[4], put_in[4], odd;
  // while the list is made: a region cell's sums within its chunk of 64, and a
  // list entry's region cell and slot
  int *const part_sum = reinterpret_cast<int *>(&list[0]);
  unsigned short *const map = reinterpret_cast<unsigned short *>(&draw[0][0]);
  static_assert(sizeof(list) >= sizeof(int) * kRegion, "the sums lie over the list");
  static_assert(sizeof(draw) >= sizeof(unsigned short) * kSpheres, "the map lies over the draws");

  // consecutive bricks to one XCD (workgroups go round the 8 in turn): its L2
  // holds the records its bricks share, phase after phase
  const int per = (nb + 7) / 8, bi = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || bi >= nb) return;
  const Brick br = bricks[bi];
  const RepDev rp = reps[br.r];
  const SweepDev sw = swp[br.r];
  const unsigned long long sweep = *sweep_base + (unsigned long long)k;
  const int par = (int)(sweep & 1ull);
  const int *cntb = cnt + (size_t)par * C + rp.coff;
  SlotRec *slot = slot_all + (size_t)(one ? par : 0) * CAP * C + rp.coff;
  const int colour = (int)((sw.order >> (4 * phase)) & 0xFu);
  const int ox = colour & 1, oy = (colour >> 1) & 1, oz = (colour >> 2) & 1;
  // The brick at once; where it or its neighbourhood holds more spheres than
  // fit (a lattice's layers, an uneven configuration), half of it after the
  // other along its longest side, and a half that does not fit cell by cell.
  int half = -1, single = -1;
  for (bool again = false;; again = true) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // as here(), for what is derived from the lane
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int x0 = br.x0, y0 = br.y0, z0 = br.z0, nx = br.nx, ny = br.ny, nz = br.nz;
    if (half >= 0) {
      const int axis = nx >= ny && nx >= nz ? 0 : (ny >= nz ? 1 : 2);
      const int n = axis == 0 ? nx : (axis == 1 ? ny : nz), first = (n + 1) / 2;
      const int skip = half ? first : 0, take = half ? n - first : first;
      x0 += axis == 0 ? skip : 0;
      y0 += axis == 1 ? skip : 0;
      z0 += axis == 2 ? skip : 0;
      nx = axis == 0 ? take : nx;
      ny = axis == 1 ? take : ny;
      nz = axis == 2 ? take : nz;
    }
    const int cells = nx * ny * nz;
    if (single >= 0) {
      const int by = here(ny), bz = here(nz);
      x0 += single / (by * bz);
      y0 += single / bz % by;
      z0 += single % bz;
      nx = ny = nz = 1;
    }
    const int na = nx * ny * nz;
    const int ry = 2 * ny + 1, rz = 2 * nz + 1, ncell = (2 * nx + 1) * ry * rz;
    const int lx = 2 * x0 + ox - 1, ly = 2 * y0 + oy - 1, lz = 2 * z0 + oz - 1;  // first cells of the region
    auto grid_cell = [&](int ix, int iy, int iz) { return cell_at[0][ix] + cell_at[1][iy] + cell_at[2][iz]; };

    // i / rz and i / ry, exact below 2^20 / rz (the float quotients' errors
    // are far below the distance to the next integer, 1 / rz at least)
    const unsigned mz = (unsigned)(1048576.0f / (float)rz) + 1u, my = (unsigned)(1048576.0f / (float)ry) + 1u;
    auto place_of = [&](int i, int &ix, int &iy, int &iz) {
      const int t = (int)((unsigned)i * mz >> 20);
      iz = i - t * rz;
      ix = (int)((unsigned)t * my >> 20);
      iy = t - ix * ry;
    };

    if (again) __syncthreads();  // the last part's lists are no longer read
    if (tid < 3 * kSide) {
      const int d = tid / kSide, i = tid - d * kSide;
      const int first = d == 0 ? lx : d == 1 ? ly : lz, g = d == 0 ? rp.gx : d == 1 ? rp.gy : rp.gz;
      const double side = d == 0 ? rp.sx : d == 1 ? rp.sy : rp.sz, shift = d == 0 ? sw.shx : d == 1 ? sw.shy : sw.shz;
      centre[d][i] = (first + i + 0.5) * side + shift;
      cell_at[d][i] = wrap_index(first + i, g) * (d == 0 ? rp.gy * rp.gz : d == 1 ? rp.gz : 1);
    }
    if (tid < 4) bin[tid] = put_in[tid] = 0;
    if (tid == 4) odd = rp.dr_max > 2.0 * fmin(rp.lx, fmin(rp.ly, rp.lz));  // steps may end outside the box
    __syncthreads();
    // prefix sums of the region's counts, a cell to a lane: within chunks of
    // 64, then over the chunks; spheres in the low 16 bits and those of
    // active cells (odd places along each axis) above.
    // All loads of a thread in flight together.
    {
      int n[kPer], v[kPer];
#pragma unroll
      for (int j = 0; j < kPer; ++j) {
        const int i = tid + j * kThreads;
        int ix, iy, iz;
        place_of(i < ncell ? i : 0, ix, iy, iz);
        n[j] = cntb[(unsigned)grid_cell(ix, iy, iz)];
        v[j] = i < ncell ? ((ix & iy & iz & 1) ? 0x10001 : 1) : 0;
      }
#pragma unroll
      for (int j = 0; j < kPer; ++j) {
        const int sum = group_inclusive_sum<64>(min(n[j], CAP) * v[j]);
        part_sum[tid + j * kThreads] = sum;
        if (lane == 63) chunk_sum[wave + 4 * j] = sum;
      }
    }
    __syncthreads();
    const int of_chunk = lane < kPer * 4 ? chunk_sum[lane] : 0, upto = group_inclusive_sum<64>(of_chunk);
    const int all = __builtin_amdgcn_readlane(upto, 63);  // a scalar: the brick's shape stays one
    const int total = all & 0xFFFF, attempts = all >> 16;
    if (total > kSpheres || attempts > kAttempts) {  // the same in every thread; not a single cell's stencil
      if (half < 0)
        half = 0;
      else
        single = 0;
      continue;
    }
#pragma unroll 1
    for (int i = tid, m = wave; i - tid < ncell; i += kThreads, m += 4) {
      const int before = __builtin_amdgcn_readlane(upto - of_chunk, __builtin_amdgcn_readfirstlane(m));
      if (i >= ncell) continue;
      int ix, iy, iz;
      place_of(i, ix, iy, iz);
      const int end = part_sum[i], begin = lane ? part_sum[i - 1] : 0;
      const int n = (end - begin) & 0xFFFF, s = before + begin, e = s & 0xFFFF, a = s >> 16;
      const bool active = ix & iy & iz & 1;
      const int c = ((ix >> 1) * ny + (iy >> 1)) * nz + (iz >> 1);
      start[i] = (unsigned short)e;
      if (active) {
        first_att[c] = (unsigned short)a;
        act_at[c] = (ix >> 1) | (iy >> 1) << 8 | (iz >> 1) << 16;
        if (n) atomicAdd(&bin[min(n, 3)], 1);
      }
#pragma unroll 1
      for (int q = 0; q < n; ++q) {
        map[e + q] = (unsigned short)(i | q << 11);
        if (active) att_cell[a + q] = (unsigned char)c;
      }
    }
    if (tid == 0) start[ncell] = (unsigned short)total;
    __syncthreads();

    // the list, a sphere to a lane
    {
      auto load = [&](int e, int &ix, int &iy, int &iz, int &at) {
        const int m = map[e];
        place_of(m & 2047, ix, iy, iz);
        at = (m >> 11) * C + grid_cell(ix, iy, iz);
        return slot[(unsigned)at];
      };
      auto place = [&](double v, int d, int i, double L) {
        const double off = v - centre[d][i], wrap = __builtin_fabs(off) > 0.5 * L ? __builtin_copysign(L, off) : 0.0;
        if (outside(v, L)) odd = 1;  // all others lie within half a side of the centre, or an edge from there
        return (float)(v - centre[d][0] - wrap);
      };
      auto put = [&](int e, const SlotRec &r, int ix, int iy, int iz, int at) {
        float4 v;
        v.x = place(r.x, 0, ix, rp.lx);
        v.y = place(r.y, 1, iy, rp.ly);
        v.z = place(r.z, 2, iz, rp.lz);
        v.w = __int_as_float(at);
        if (ix & iy & iz & 1) {
          const int a = first_att[((ix >> 1) * ny + (iy >> 1)) * nz + (iz >> 1)] + (map[e] >> 11);
          pos[0][a] = r.x;
          pos[1][a] = r.y;
          pos[2][a] = r.z;
          v.w = __int_as_float(r.id);
        }
        list[e] = v;
      };
#pragma unroll 1
      for (int e0 = tid; e0 < total; e0 += kRecs * kThreads) {
        int ix[kRecs], iy[kRecs], iz[kRecs], at[kRecs];
        SlotRec rec[kRecs];
#pragma unroll
        for (int j = 0; j < kRecs; ++j) {
          const int e = e0 + j * kThreads;
          rec[j] = load(e < total ? e : e0, ix[j], iy[j], iz[j], at[j]);
        }
#pragma unroll
        for (int j = 0; j < kRecs; ++j) {
          const int e = e0 + j * kThreads;
          if (e < total) put(e, rec[j], ix[j], iy[j], iz[j], at[j]);
        }
      }
    }
    auto region_cell = [&](int ix, int iy, int iz) { return ((2 * ix + 1) * ry + 2 * iy + 1) * rz + 2 * iz + 1; };
    auto active_at = [&](int c, int &ix, int &iy, int &iz) {
      const int at = act_at[c];
      ix = at & 0xFF;
      iy = at >> 8 & 0xFF;
      iz = at >> 16;
    };
    // active cells, those with most occupants first, so that few waves go
    // round more than once
    const int n3 = __builtin_amdgcn_readfirstlane(bin[3]), n2 = __builtin_amdgcn_readfirstlane(bin[2]),
              n1 = __builtin_amdgcn_readfirstlane(bin[1]);
    if (tid < na) {
      int ix, iy, iz;
      active_at(tid, ix, iy, iz);
      const int i = region_cell(ix, iy, iz), nc = min(start[i + 1] - start[i], 3);
      if (nc) order[atomicAdd(&put_in[nc], 1) + (nc == 3 ? 0 : nc == 2 ? n3 : n3 + n2)] = (unsigned char)tid;
    }
    __syncthreads();

    // a lane to an attempt: its occupant and its displacement's draws
    for (int a = tid; a < attempts; a += kThreads) {
      const int c = att_cell[a], a0 = first_att[c], t = a - a0;
      int ix, iy, iz;
      active_at(c, ix, iy, iz);
      const int i = region_cell(ix, iy, iz), e0 = start[i], nc = start[i + 1] - e0;
      const int cid = ((2 * (x0 + ix) + ox) * rp.gy + 2 * (y0 + iy) + oy) * rp.gz + 2 * (z0 + iz) + oz;
      uint32_t w[4];
      const uint32_t k0 = (uint32_t)here((int)rp.k0), k1 = (uint32_t)here((int)rp.k1);
      philox4x32_10((uint32_t)cid, (uint32_t)t, (uint32_t)sweep, (uint32_t)(sweep >> 32), k0, k1, w);
      const int pick = (int)occupant_pick(w[0], (uint32_t)nc, (uint32_t)cid, (uint32_t)t, sweep, k0, k1);
      draw[0][a] = w[1];
      draw[1][a] = w[2];
      draw[2][a] = w[3];
      // the occupant of that rank in ascending particle id
      int q = 0;
#pragma unroll 1
      for (int m = 0; m < nc; ++m) {
        const int id = __float_as_int(list[e0 + m].w);
        int rank = 0;
#pragma unroll 1
        for (int o = 0; o < nc; ++o) rank += __float_as_int(list[e0 + o].w) < id ? 1 : 0;
        q = rank == pick ? m : q;
      }
      slot_of[a] = (unsigned char)q;
    }
    __syncthreads();

    // 4 lanes to an active cell: its attempts one after another.  Lane d < 3
    // of the 4 works out where an attempt leads along axis d.
    const int ql = tid & 3, axis = ql < 3 ? ql : 0;
    const bool any_odd = __builtin_amdgcn_readfirstlane(odd) != 0;
    const double L = axis == 0 ? rp.lx : axis == 1 ? rp.ly : rp.lz;
    const double shift = axis == 0 ? sw.shx : axis == 1 ? sw.shy : sw.shz;
    const double inv_side = axis == 0 ? rp.ix : axis == 1 ? rp.iy : rp.iz;
    const int g = axis == 0 ? rp.gx : axis == 1 ? rp.gy : rp.gz;
    const int first = axis == 0 ? lx : axis == 1 ? ly : lz;
    const double frame0 = centre[axis][0];
    auto of_axis = [](float v, int d) {  // lane d's v in all 4 lanes
      const int b = __float_as_int(v);
      return __int_as_float(d == 0   ? __builtin_amdgcn_update_dpp(0, b, 0x00, 0xf, 0xf, true)
                            : d == 1 ? __builtin_amdgcn_update_dpp(0, b, 0x55, 0xf, 0xf, true)
                                     : __builtin_amdgcn_update_dpp(0, b, 0xaa, 0xf, 0xf, true));
    };
    for (int quad = tid >> 2; quad < n3 + n2 + n1; quad += kThreads / 4) {
      const int c = order[quad];
      int ix, iy, iz;
      active_at(c, ix, iy, iz);
      const int i0 = region_cell(ix, iy, iz), e0 = start[i0], a0 = first_att[c];
      int nc = start[i0 + 1] - e0;
      // the stencil's 9 rows of 3 cells: rows ql and ql + 4 are this lane's, and
      // every fourth entry of the last, walked as one run of `len` entries
      auto row_at = [&](int row) {
        const int base = i0 + ((row / 3 - 1) * ry + row % 3 - 1) * rz, b = start[base - 1];
        return make_int2(b, start[base + 2] - b);
      };
      const int2 r0 = row_at(ql), r1 = row_at(ql + 4), r2 = row_at(8);
      const int b0 = r0.x, b1 = r1.x, b2 = r2.x, l0 = r0.y, l01 = l0 + r1.y, len = l01 + ((r2.y + 3 - ql) >> 2);
      const int p1 = b1 - l0, p2 = b2 + ql - 4 * l01;
      int T = len + __shfl_xor(len, 1, 4);
      T += __shfl_xor(T, 2, 4);
      if (T > lcap) {
        // the capacity of the other kernels' stencil list, which holds a cell
        // once where an axis has two (the region has it before and after)
        int once = 0;
#pragma unroll 1
        for (int j = 0; j < 27; ++j) {
          const int dx = j / 9 - 1, dy = j / 3 % 3 - 1, dz = j % 3 - 1, i = i0 + (dx * ry + dy) * rz + dz;
          if (stencil_axis_ok(dx, rp.gx) && stencil_axis_ok(dy, rp.gy) && stencil_axis_ok(dz, rp.gz))
            once += start[i + 1] - start[i];
        }
        if (once > lcap) {
          if (ql == 0) atomicOr(err, kErrListFull);
          nc = 0;
        }
      }
      unsigned n_acc = 0, n_left = 0, moved = 0;
#pragma unroll 1
      for (int t = 0; t < nc; ++t) {
        const int a = a0 + t, q = slot_of[a], self = e0 + q;
        const double to = wrap_once(pos[axis][a0 + q] + (u32_unit_closed(draw[axis][a]) - 0.5) * rp.dr_max, L);
        const int place = 2 * (axis == 0 ? ix : axis == 1 ? iy : iz) + 1;  // in the region
        const bool stays = shifted_cell(to, shift, L, inv_side, g) == first + place;
        if ((__ballot(!stays) >> (lane & ~3) & 0x7ull) != 0ull) {
          ++n_left;
          continue;
        }
        const double off = to - centre[axis][place];
        const float f = (float)(to - frame0 - (__builtin_fabs(off) > 0.5 * L ? __builtin_copysign(L, off) : 0.0));
        const float fx = of_axis(f, 0), fy = of_axis(f, 1), fz = of_axis(f, 2);
        auto entry = [b0, p1, p2, l0, l01](int u) {
          const int p = u < l0 ? b0 : p1, near = u + p, last = 4 * u + p2;
          return u < l01 ? near : last;
        };
        float nearest = 9.0f;
#pragma unroll 1
        for (int u0 = 0; u0 < len; u0 += kRead) {
          float4 v[kRead];
          int e[kRead];
#pragma unroll
          for (int u = 0; u < kRead; ++u) {
            e[u] = u0 + u < len ? entry(u0 + u) : self;
            v[u] = list[e[u]];
          }
#pragma unroll
          for (int u = 0; u < kRead; ++u) {
            const float dx = fx - v[u].x, dy = fy - v[u].y, dz = fz - v[u].z;
            const float s = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
            nearest = e[u] == self ? nearest : fminf(nearest, s);
          }
        }
        bool hit = nearest < 1.0f - kBand;
        const bool undecided = any_odd || (!hit && nearest < 1.0f + kBand);
        if (__any(undecided)) {
          const double qx = __shfl(to, 0, 4), qy = __shfl(to, 1, 4), qz = __shfl(to, 2, 4);
          if (undecided) hit = false;
#pragma unroll 1
          for (int u = undecided ? 0 : len; u < len; ++u) {
            const int e = entry(u);
            double bx, by, bz;
            if (e >= e0 && e < e0 + nc) {  // an occupant of this cell, moved or not
              bx = pos[0][a0 + e - e0];
              by = pos[1][a0 + e - e0];
              bz = pos[2][a0 + e - e0];
            } else {
              const SlotRec *r = slot + __float_as_int(list[e].w);
              bx = r->x;
              by = r->y;
              bz = r->z;
            }
            hit |= e != self && dist2(qx, qy, qz, bx, by, bz, rp.lx, rp.ly, rp.lz) < 1.0;
          }
        }
        if ((__ballot(hit) >> (lane & ~3) & 0xFull) != 0ull) continue;
        if (ql < 3) {
          pos[axis][a0 + q] = to;
          reinterpret_cast<float *>(&list[self])[axis] = f;
        }
        wave_lds_sync();
        moved |= 1u << q;
        ++n_acc;
      }
      // the spheres that moved, to their records and by-id positions
      const int cid = ((2 * (x0 + ix) + ox) * rp.gy + 2 * (y0 + iy) + oy) * rp.gz + 2 * (z0 + iz) + oz;
#pragma unroll 1
      for (int q = ql; q < nc; q += 4) {
        if (!(moved >> q & 1u)) continue;
        SlotRec *r = slot + (size_t)q * C + cid;
        const int g = rp.poff + __float_as_int(list[e0 + q].w);
        const double px = pos[0][a0 + q], py = pos[1][a0 + q], pz = pos[2][a0 + q];
        store_through(&r->x, px);
        store_through(&r->y, py);
        store_through(&r->z, pz);
        store_through(&x[g], px);
        store_through(&y[g], py);
        store_through(&z[g], pz);
      }
      if (ql == 0) {
        const int ai = rp.aoff + ((x0 + ix) * (rp.gy >> 1) + y0 + iy) * (rp.gz >> 1) + z0 + iz;
        if (n_acc) atomicAdd(&cacc[ai], n_acc);
        if (n_left) atomicAdd(&cleft[ai], n_left);
      }
    }
    if (half < 0) break;
    if (single >= 0 && ++single < cells) continue;
    single = -1;
    if (++half == 2) break;
  }
}

// Ends of n active cells along an axis in `parts` parts as even as can be.
std::vector<int> axis_parts(int n, int parts) {
  std::vector<int> end(parts);
  for (int p = 0; p < parts; ++p) end[p] = (int)((long)n * (p + 1) / parts);
  return end;
}

}  // namespace

namespace hsmc {

bool bricks_run(const hsmc_gpu_ctx *ctx) { return !ctx->tune_set && ctx->n_bricks > 0; }

// The bricks of every replica, small enough for its density (a brick that
// does not fit all the same goes cell by cell).
int build_bricks(hsmc_gpu_ctx *ctx) {
  ctx->n_bricks = 0;
  if (ctx->Atot < kBrickCells) return HSMC_OK;
  std::vector<Brick> v;
  long active = 0;  // without the padding of small replicas
  for (int r = 0; r < ctx->R; ++r) {
    const RepHost &h = ctx->reps[r];
    active += (long)h.gx * h.gy * h.gz / 8;
    // the shape that costs least: a workgroup's own work and its region's
    const double in_cell = h.p.n_part / ((double)h.gx * h.gy * h.gz);
    auto fits = [&](long cells, int room) {  // with room for uneven density
      const double mean = in_cell * cells;
      return mean + 4.0 * std::sqrt(mean) <= room;
    };
    const int hx = h.gx / 2, hy = h.gy / 2, hz = h.gz / 2;
    int px = hx, py = hy, pz = hz;  // single cells
    // cells of an axis in less than 32 diameters, also when the box has grown
    // to the next grid
    auto frame_fits = [](int b, int g) { return (2 * b + 1) * (1.0 + 2.0 / g) < 32.0; };
    double best = INFINITY;
    for (int bz = 1; bz <= std::min(hz, kSide / 2); ++bz)
      for (int by = 1; by <= std::min({hy, kSide / 2, kActive / bz}); ++by)
        for (int bx = 1; bx <= std::min({hx, kSide / 2, kActive / (bz * by)}); ++bx) {
          const long region = (2L * bx + 1) * (2 * by + 1) * (2 * bz + 1);
          if (!frame_fits(bx, h.gx) || !frame_fits(by, h.gy) || !frame_fits(bz, h.gz)) continue;
          if (region > kRegion || !fits(region, kSpheres) || !fits((long)bx * by * bz, kAttempts))
            continue;
          const long nx = (hx + bx - 1) / bx, ny = (hy + by - 1) / by, nz = (hz + bz - 1) / bz;
          const double cost = (double)nx * ny * nz * (400.0 + region);
          if (cost < best) best = cost, px = nx, py = ny, pz = nz;
        }
    const std::vector<int> ex = axis_parts(hx, px), ey = axis_parts(hy, py), ez = axis_parts(hz, pz);
    int x0 = 0;
    for (int x1 : ex) {
      int y0 = 0;
      for (int y1 : ey) {
        int z0 = 0;
        for (int z1 : ez) {
          v.push_back(Brick{r, x0, y0, z0, x1 - x0, y1 - y0, z1 - z0, 0});
          z0 = z1;
        }
        y0 = y1;
      }
      x0 = x1;
    }
  }
  if (active < kBrickMean * (long)v.size()) return HSMC_OK;  // cell by cell
  if (v.size() > ctx->brick_alloc) {
    (void)hipFree(ctx->d_bricks);
    ctx->d_bricks = nullptr;
    ctx->brick_alloc = 0;
    const size_t want = v.size() + v.size() / 8;
    HSMC_HIP(ctx, hipMalloc(&ctx->d_bricks, sizeof(Brick) * want));
    ctx->brick_alloc = want;
  }
  HSMC_HIP(ctx, hipMemcpy(ctx->d_bricks, v.data(), sizeof(Brick) * v.size(), hipMemcpyHostToDevice));
  ctx->n_bricks = (int)v.size();
  return HSMC_OK;
}

void enqueue_brick_phase(hsmc_gpu_ctx *ctx, int phase, int k, hipStream_t s) {
  const int nb = ctx->n_bricks;
  hipLaunchKernelGGL(ctx->cap == 8 ? k_brick_phase<8> : k_brick_phase<16>, dim3((unsigned)((nb + 7) / 8 * 8)),
                     dim3(kThreads), 0, s, ctx->d_sweep, ctx->d_swp, ctx->d_reps, ctx->d_bricks, nb,
                     ctx->R == 1 ? 1 : 0, phase, k, ctx->lcap, ctx->d_x, ctx->d_y, ctx->d_z, ctx->d_cnt,
                     (int)ctx->Ctot, ctx->d_slot, ctx->d_cacc, ctx->d_cleft, ctx->d_err);
}

}  // namespace hsmc
