// device_common.h -- FP64 distance arithmetic, cell indexing and the
// Philox4x32-10 counter RNG shared by every kernel of libhsmc_gpu.
//
// All FP64 expressions here are evaluated without contraction (the TU is
// built with -ffp-contract=off and the pragma below), in the reference's
// order (moves.c:400-431), so every overlap decision and histogram bin is
// rounded exactly as the reference rounds it.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#pragma clang fp contract(off)

namespace hsmc {

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11): 10 rounds of the
// multiply-xor bijection with the Weyl key schedule.
__host__ __device__ __forceinline__ void philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2,
                                                       uint32_t c3, uint32_t k0, uint32_t k1,
                                                       uint32_t out[4]) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    if (r) {
      k0 += 0x9E3779B9u;
      k1 += 0xBB67AE85u;
    }
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
    const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0;
    const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
    c0 = n0;
    c1 = (uint32_t)p1;
    c2 = n2;
    c3 = (uint32_t)p0;
  }
  out[0] = c0;
  out[1] = c1;
  out[2] = c2;
  out[3] = c3;
}

// rng_get_double (rng.c:29-31): a 32-bit draw divided by 2^32-1, in [0,1].
// 1/(2^32 - 1) is the geometric series 2^-32 + 2^-64 + 2^-96 + ..., so one
// fused multiply-add, which rounds u (2^-32 + 2^-64) + u 2^-96 once, gives
// the correctly rounded quotient: the terms left out are below 2^-128 u, and
// every one of the 2^32 values of u was compared with the IEEE division.  A
// product and an FMA in place of a division's dozen FP64 instructions.
__host__ __device__ __forceinline__ double u32_unit_closed(uint32_t u) {
  const double x = (double)u;
  return __builtin_fma(x, 0x1.00000001p-32, x * 0x1p-96);
}

// Occupant pick of the checkerboard sweep: rng_get_int's rule (rng.c:34-36,
// gsl_rng_uniform_int) applied to the sweep's Philox stream.  `first` is word
// 0 of attempt t's block (counter cell, t, sweep); k = first / scale with
// scale = (2^32 - 1) / n, and a k >= n is drawn again from the block with
// counter word 1 = t | (retry << 16), retry = 1, 2, ...  Uniform on [0, n)
// for any n in [1, 2^32 - 1] and t < 2^16.
__host__ __device__ __forceinline__ uint32_t occupant_pick(uint32_t first, uint32_t n,
                                                           uint32_t cell, uint32_t t,
                                                           unsigned long long sweep, uint32_t k0,
                                                           uint32_t k1) {
  const uint32_t scale = 0xFFFFFFFFu / n;
  uint32_t k = first / scale;
  for (uint32_t rr = 1; k >= n; ++rr) {
    uint32_t w[4];
    philox4x32_10(cell, t | (rr << 16), (uint32_t)sweep, (uint32_t)(sweep >> 32), k0, k1, w);
    k = w[0] / scale;
  }
  return k;
}

// Minimum image of one component (moves.c:419-424): d - L above half a box,
// d + L below minus half a box.  Both candidates are computed and one is
// selected, so the compiler emits selects rather than branches.
__host__ __device__ __forceinline__ double min_image(double d, double L, double half) {
  const double dm = d - L, dp = d + L;
  return d > half ? dm : (d < -half ? dp : d);
}

// |min_image(d, L, L/2)| in two instructions (min_image's selects take
// eight).  L/2 is exact.  For |d| <= L/2, L - |d| >= L/2 >= |d| and rounding
// is monotone, so the minimum is |d|; for |d| > L/2, L - |d| < L/2 < |d| and
// the minimum is L - |d|, which rounds to the negative of |d| - L.  So it is
// the same double up to its sign, which a squared distance does not see, for
// every d (also beyond L, infinite or NaN).  With the draw's division and
// the search grids' divisions gone as well: a sweep at N = 32000 46.2 -> 44.2
// us, at N = 256 43.5 -> 40.0 us; one stratified Widom sample at N = 108000
// 308 -> 291 us, one learned sample 375 -> 350 us, one g(r) sample at
// N = 32000 441 -> 402 us.
__host__ __device__ __forceinline__ double image_mag(double d, double L) {
  const double a = __builtin_fabs(d);
  return __builtin_fmin(a, L - a);
}

// Squared distance of the reference's compute_dist with unit scale
// (moves.c:414-427): a - b per axis, minimum image, dx*dx+dy*dy+dz*dz.
// dr < 1 <=> dr^2 < 1 for correctly rounded sqrt, so overlap tests use it.
__host__ __device__ __forceinline__ double dist2(double ax, double ay, double az, double bx,
                                                 double by, double bz, double lx, double ly,
                                                 double lz) {
  const double dx = image_mag(ax - bx, lx);
  const double dy = image_mag(ay - by, ly);
  const double dz = image_mag(az - bz, lz);
  return dx * dx + dy * dy + dz * dz;
}

// compute_dist with a scale factor (moves.c:405-427): dx = (a-b)*sf and a
// box of L*sf, half box (L*sf)/2.
__host__ __device__ __forceinline__ double dist2_scaled(double ax, double ay, double az,
                                                        double bx, double by, double bz,
                                                        double lx, double ly, double lz,
                                                        double sf) {
  const double dx = image_mag((ax - bx) * sf, lx * sf);
  const double dy = image_mag((ay - by) * sf, ly * sf);
  const double dz = image_mag((az - bz) * sf, lz * sf);
  return dx * dx + dy * dy + dz * dz;
}

// apply_pbc for one coordinate (moves.c:215-226): a single wrap (selected,
// not branched, as in min_image).
__host__ __device__ __forceinline__ double wrap_once(double x, double L) {
  const double xm = x - L, xp = x + L;
  return x > L ? xm : (x < 0.0 ? xp : x);
}

// Cell of coordinate x on a grid of g cells of side `side` whose origin is
// shifted by `shift` in [0, side): t = x - shift (wrapped), (int)(t * (1/side)),
// clamped to g-1 at t == L.  Multiplying by the rounded reciprocal moves each
// cell edge by a few ulp at most, so every cell stays wider than the grid's
// minimum side of 1 + 1e-9 diameters.
__host__ __device__ __forceinline__ int shifted_cell(double x, double shift, double L,
                                                     double inv_side, int g) {
  const double t0 = x - shift, t1 = t0 + L;
  const double t = t0 < 0.0 ? t1 : t0;
  const int c = (int)(t * inv_side);
  return c < g ? c : g - 1;
}

// The cell of that grid a sphere is filed in.  A position a side and more
// below the shifted origin's image is left of the grid (steps wider than four
// box edges lead there: the wrap is a single one) and goes to the first cell.
__host__ __device__ __forceinline__ int filed_cell(double x, double shift, double L,
                                                   double inv_side, int g) {
  const int c = shifted_cell(x, shift, L, inv_side, g);
  return c < 0 ? 0 : c;
}

// Cell of coordinate x on an unshifted grid (cell_part_idx, cell_list.c:244-246),
// clamped into [0, g-1].
__host__ __device__ __forceinline__ int plain_cell(double x, double side, int g) {
  int c = (int)(x / side);
  if (c >= g) c = g - 1;
  if (c < 0) c = 0;
  return c;
}

// The same on a search grid (the reference has none of these): a product
// with the rounded reciprocal in place of a division's dozen FP64
// instructions.  It moves each cell edge by a few ulp at most, far inside
// the margin by which every search grid's side exceeds its cutoff, so the
// 27 cells around a point still hold every sphere within the cutoff.
__host__ __device__ __forceinline__ int search_cell(double x, double inv_side, int g) {
  int c = (int)(x * inv_side);
  if (c >= g) c = g - 1;
  if (c < 0) c = 0;
  return c;
}

// Per-axis neighbour offsets of the 27-cell stencil that are distinct on a
// periodic grid of g cells: g >= 3 -> {-1,0,1}; g == 2 -> {0,1}; g == 1 -> {0}.
__host__ __device__ __forceinline__ bool stencil_axis_ok(int d, int g) {
  if (g >= 3) return true;
  if (g == 2) return d != -1;
  return d == 0;
}

// The 27-cell stencil in order of distance class |dx| + |dy| + |dz| (own
// cell, faces, edges, corners; lexicographic within a class), for scans
// that can stop at the first sphere found near a point.  Entry k of the
// order is the lexicographic index t = (dx+1)*9 + (dy+1)*3 + (dz+1), kept
// in 5 bits at position k % 9 of word k / 9; the words are built at compile
// time, so a lane finds its offset with a few shifts.
namespace detail {
constexpr uint64_t stencil_order_word(int w) {
  uint64_t word = 0;
  int k = 0;
  for (int cls = 0; cls <= 3; ++cls)
    for (int t = 0; t < 27; ++t) {
      const int ox = t / 9 - 1, oy = (t / 3) % 3 - 1, oz = t % 3 - 1;
      const int c = (ox < 0 ? -ox : ox) + (oy < 0 ? -oy : oy) + (oz < 0 ? -oz : oz);
      if (c != cls) continue;
      if (k / 9 == w) word |= (uint64_t)t << (5 * (k % 9));
      ++k;
    }
  return word;
}
}  // namespace detail

// Offset j in [0, 27) of that order; returns its distance class.
__host__ __device__ __forceinline__ int stencil_by_distance(int j, int &dx, int &dy, int &dz) {
  constexpr uint64_t w0 = detail::stencil_order_word(0), w1 = detail::stencil_order_word(1),
                     w2 = detail::stencil_order_word(2);
  const uint64_t word = j < 9 ? w0 : (j < 18 ? w1 : w2);
  const int t = (int)((word >> (5 * (j % 9))) & 31u);
  dx = t / 9 - 1;
  dy = (t / 3) % 3 - 1;
  dz = t % 3 - 1;
  return (dx < 0 ? -dx : dx) + (dy < 0 ? -dy : dy) + (dz < 0 ? -dz : dz);
}

__host__ __device__ __forceinline__ int wrap_index(int i, int g) {
  if (i < 0) i += g;
  else if (i >= g) i -= g;
  return i;
}

// LDS written by one lane of a wave is read by its others after this.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Inclusive sum of v over each group of LPC (32 or 64) consecutive lanes of
// a full wave, in DPP moves with no LDS round trip: shifts by 1, 2, 4 and 8
// within each row of 16 lanes, then lane 15 of each even row added to the
// row above it (the two halves of a 32-lane group) and, for 64-lane groups,
// lane 31 added to rows 2 and 3.  A shifted-in lane outside the row reads 0.
template <int LPC>
__device__ __forceinline__ int group_inclusive_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1, 3
  if constexpr (LPC == 64)
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2, 3
  return v;
}

}  // namespace hsmc
