// sweep_draws.h -- what one checkerboard sweep of a replica draws before any
// move, shared by the launched and the resident sweep kernels.
#pragma once
#include "ctx.h"
#include "device_common.h"

namespace hsmc {

// Vector store at agent scope: written through the XCD's L2 (the next
// phase's workgroups read it from other XCDs).
__device__ __forceinline__ void store_through(double *p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Shift of the sweep grid for one sweep: 3 uniform draws in [0, side).
__device__ __forceinline__ void sweep_shift(const RepDev &rp, unsigned long long sweep,
                                            double &shx, double &shy, double &shz) {
  uint32_t u[4];
  philox4x32_10(0xFFFFFFFFu, 0u, (uint32_t)sweep, (uint32_t)(sweep >> 32), rp.k0, rp.k1, u);
  shx = ((double)u[0] * 0x1p-32) * rp.sx;
  shy = ((double)u[1] * 0x1p-32) * rp.sy;
  shz = ((double)u[2] * 0x1p-32) * rp.sz;
}

// Order of the 8 sublattices in one sweep: a Fisher-Yates order of 0..7
// drawn from one Philox block, kept as 8 nibbles (nibble p = sublattice of
// phase p).
__device__ __forceinline__ uint32_t sweep_order(const RepDev &rp, unsigned long long sweep) {
  uint32_t u[4];
  philox4x32_10(0xFFFFFFFEu, 0u, (uint32_t)sweep, (uint32_t)(sweep >> 32), rp.k0, rp.k1, u);
  uint32_t pk = 0x76543210u;
#pragma unroll
  for (int h = 0; h < 7; ++h) {
    const int i = 7 - h;
    const uint32_t half = (u[h >> 1] >> (16 * (h & 1))) & 0xFFFFu;
    const int j = (int)((half * (uint32_t)(i + 1)) >> 16);
    const uint32_t vi = (pk >> (4 * i)) & 0xFu, vj = (pk >> (4 * j)) & 0xFu;
    pk &= ~((0xFu << (4 * i)) | (0xFu << (4 * j)));
    pk |= (vi << (4 * j)) | (vj << (4 * i));
  }
  return pk;
}

}  // namespace hsmc
