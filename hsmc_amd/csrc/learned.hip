// learned.hip -- learned Widom proposal (no counterpart in the reference,
// whose insertions are uniform: compute_widom_chem_pot.c:44-80).
//
// The box is divided into M^3 voxels of side ~0.25 sigma.  Each voxel gets a
// descriptor -- the sorted distances from its centre to its 12 nearest sphere
// centres (FP32) -- and a score f_v from a 12->64->64->1 ReLU network whose
// weights are BF16 and whose products run on the MFMA units with FP32
// accumulation.  Insertions are drawn from q_v = mix * softmax(f)_v +
// (1 - mix)/V by systematic sampling (insertion i falls in the voxel whose
// cumulative-mass interval holds (i + u0)/n: voxel v receives floor(n q_v)
// or one more, with mean exactly n q_v) and placed uniformly in their voxel;
// the overlap test is the exact FP64 one.  The estimate
// P = (1/(V n)) sum_hits 1/q_v of the insertion probability is unbiased for
// any q with q_v > 0, so plain uniform insertion stays the reference.
//
// The network is trained on the GPU by the kernels below (forward, backward,
// Adam) on uniform insertions: input the descriptor of the voxel holding the
// point, target -beta * max(0, 1 - d_min) with d_min the point's distance to
// the nearest centre.
#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "ctx.h"
#include "device_common.h"
#include "hsmc_gpu.h"

using namespace hsmc;

namespace {

constexpr int NIN = HSMC_MLP_IN;       // 12 descriptor entries
constexpr int KIN = 16;                // padded to the MFMA K
constexpr int NH = HSMC_MLP_HIDDEN;    // 64
constexpr int OW1 = 0, OB1 = OW1 + NIN * NH, OW2 = OB1 + NH, OB2 = OW2 + NH * NH,
              OW3 = OB2 + NH, OB3 = OW3 + NH, NPARAM = OB3 + 1;
static_assert(NPARAM == HSMC_MLP_NPARAM, "parameter layout");

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// round-to-nearest-even FP32 -> BF16 (finite inputs)
__host__ __device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// Network as the kernels read it.  Every layer is computed transposed (units
// by rows of the batch): the weights are the MFMA's A operand, a batch row
// is a column, and the result of one layer (lane l: column l % 16, units
// 4 (l / 16) .. + 3 of a 16-unit tile) is the B operand of the next layer's
// 16-unit K step as it stands, so activations never leave the registers.
// The weights are stored in the order the lanes read them, 8 or 16 bytes a
// lane, the biases as the 4 units a lane holds.  With l16 = l % 16 and
// g4 = l / 16:
//   W1[t][l][i]     = w1[k = 4 g4 + i][unit 16 t + l16] (zero for k >= NIN)
//   W2F[o][m][l][i] = w2[in 16 (2 m + i / 4) + 4 g4 + i % 4][out 16 o + l16]
//   W2B[t][m][l][i] = w2[in 16 t + l16][out 16 (2 m + i / 4) + 4 g4 + i % 4]
struct __attribute__((aligned(16))) MlpDev {
  uint16_t W1[4][64][4];
  uint16_t W2F[4][2][64][8];
  uint16_t W2B[4][2][64][8];
  float b1[NH], b2[NH], w3[NH], b3, pad[3];
};

// Store parameter i of the packed order (value w) where the kernels read it.
__device__ __forceinline__ void put_param(MlpDev *net, int i, float w) {
  if (i < OB1) {
    const int k = i / NH, u = i % NH;
    net->W1[u >> 4][(k >> 2) * 16 + (u & 15)][k & 3] = f2bf(w);
  } else if (i < OW2) {
    net->b1[i - OB1] = w;
  } else if (i < OB2) {
    const int in = (i - OW2) / NH, out = (i - OW2) % NH;
    const uint16_t v = f2bf(w);
    net->W2F[out >> 4][in >> 5][((in >> 2) & 3) * 16 + (out & 15)][((in >> 4) & 1) * 4 + (in & 3)] = v;
    net->W2B[in >> 4][out >> 5][((out >> 2) & 3) * 16 + (in & 15)][((out >> 4) & 1) * 4 + (out & 3)] = v;
  } else if (i < OW3) {
    net->b2[i - OB2] = w;
  } else if (i < OB3) {
    net->w3[i - OW3] = w;
  } else {
    net->b3 = w;
  }
}

__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x4 to_bf16x4(f32x4 v) {
  bf16x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = (short)f2bf(v[i]);
  return r;
}

// A lane's share of the forward weights.
struct NetRegs {
  bf16x4 w1[4], w2[4][4];
  f32x4 b1[4], b2[4], w3[4];
  float b3;
  __device__ __forceinline__ explicit NetRegs(const MlpDev *__restrict__ n) {
    const int lane = threadIdx.x & 63, g4 = lane >> 4;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      w1[t] = *reinterpret_cast<const bf16x4 *>(n->W1[t][lane]);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        w2[t][2 * m] = *reinterpret_cast<const bf16x4 *>(&n->W2F[t][m][lane][0]);
        w2[t][2 * m + 1] = *reinterpret_cast<const bf16x4 *>(&n->W2F[t][m][lane][4]);
      }
      b1[t] = *reinterpret_cast<const f32x4 *>(&n->b1[16 * t + 4 * g4]);
      b2[t] = *reinterpret_cast<const f32x4 *>(&n->b2[16 * t + 4 * g4]);
      w3[t] = *reinterpret_cast<const f32x4 *>(&n->w3[16 * t + 4 * g4]);
    }
    b3 = n->b3;
  }
};

// Forward pass of 16 rows: x is the lane's 4 inputs 4 g4 .. + 3 of row l16.
// Returns the network's value of row l16 (in every lane of that row) and the
// activations of the two hidden layers (h1 as BF16, h2 in FP32).  The output
// layer sums, for each column class c = unit % 16, the 4 products in tile
// order, then the 16 sums pairwise (c ^ 1, c ^ 2, c ^ 4, c ^ 8).
__device__ __forceinline__ float forward_tile(const NetRegs &n, bf16x4 x, bf16x4 h1[4],
                                              f32x4 h2[4]) {
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    f32x4 d = mfma16(n.w1[t], x, zero);
#pragma unroll
    for (int i = 0; i < 4; ++i) d[i] = fmaxf(d[i] + n.b1[t][i], 0.f);
    h1[t] = to_bf16x4(d);
  }
  f32x4 p = zero;
#pragma unroll
  for (int o = 0; o < 4; ++o) {
    f32x4 acc = zero;
#pragma unroll
    for (int k = 0; k < 4; ++k) acc = mfma16(n.w2[o][k], h1[k], acc);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      h2[o][i] = fmaxf(acc[i] + n.b2[o][i], 0.f);
      p[i] += h2[o][i] * n.w3[o][i];
    }
  }
  float v = (p[0] + p[1]) + (p[2] + p[3]);
  v += __shfl_xor(v, 16, 64);
  v += __shfl_xor(v, 32, 64);
  return v + n.b3;
}

// The lane's 4 inputs of a training or query row from memory.
__device__ __forceinline__ bf16x4 load_x(const float *__restrict__ Xg, long row, bool valid) {
  const int g4 = (threadIdx.x & 63) >> 4;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (valid && g4 < NIN / 4) v = *reinterpret_cast<const f32x4 *>(Xg + row * NIN + 4 * g4);
  return to_bf16x4(v);
}

// Sum over the 16 lanes of each DPP row, valid in the row's lane 15.
__device__ __forceinline__ float row_sum(float v) {
  auto add = [](float a, int b) { return a + __builtin_bit_cast(float, b); };
  v = add(v, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x111, 0xf, 0xf, true));
  v = add(v, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x112, 0xf, 0xf, true));
  v = add(v, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x114, 0xf, 0xf, true));
  v = add(v, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x118, 0xf, 0xf, true));
  return v;
}

// ---- forward / backward over a batch of training rows ----------------------
// A workgroup takes 64 rows at a time, each of its 4 waves 16 of them through
// the forward pass and back to the first layer in registers; the weight
// gradients contract over the 64 rows, from activations laid out by unit in
// LDS, a 16-unit strip of dW2 and of dW1 per wave.  A workgroup keeps its
// sums in registers over all its rows and stores them once, at its own row
// of `part` (NPARAM gradients, then the sum of squared errors), which
// k_reduce_grad adds up in a fixed order: no atomics, so training is
// reproducible.  Latency-bound (64 workgroups at a batch of 4096): 6.9 us, and
// 4.4 us for k_reduce_grad.  One wave per 64 rows through LDS, with 4993 atomics
// each, took 27.9 us, and its Adam kernel 4.7 us.
constexpr int kGradStride = NPARAM + 7;  // one row of part, in floats (NPARAM + 1 used)
constexpr int kGradBlocks = 256;         // workgroups at most

__global__ void __launch_bounds__(256)
k_mlp_train_step(const MlpDev *__restrict__ net, const float *__restrict__ Xg,
                 const float *__restrict__ Tg, int n, float inv_batch, float *__restrict__ part) {
  constexpr int LD = 72;  // 64 rows and 8 of padding: 16-byte reads on different banks
  __shared__ __attribute__((aligned(16))) uint16_t H1[NH][LD], D2[NH][LD], D1[NH][LD], XT[KIN][LD];
  __shared__ float red[3][4][NH], red2[2][4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, l16 = lane & 15, g4 = lane >> 4;
  const NetRegs nr(net);
  bf16x4 w2b[4][4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      w2b[t][2 * m] = *reinterpret_cast<const bf16x4 *>(&net->W2B[t][m][lane][0]);
      w2b[t][2 * m + 1] = *reinterpret_cast<const bf16x4 *>(&net->W2B[t][m][lane][4]);
    }
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 gw2[4], gw1 = zero, g3[4], gb2[4], gb1[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) gw2[t] = g3[t] = gb2[t] = gb1[t] = zero;
  float sq = 0.f, sdy = 0.f;
  const int col = w * 16 + l16;  // this lane's row of the 64
  for (long row0 = (long)blockIdx.x * 64; row0 < n; row0 += (long)gridDim.x * 64) {
    const long row = row0 + col;
    const bool valid = row < n;
    const bf16x4 x = load_x(Xg, row, valid);
    bf16x4 h1[4];
    f32x4 h2[4];
    const float y = forward_tile(nr, x, h1, h2);
    const float e = valid ? y - Tg[row] : 0.f;
    const float dy = 2.f * e * inv_batch;
    sq += e * e;
    sdy += dy;
    // dW3 = H2 dy; dH2 = dy w3 where H2 > 0; db2 = dH2
    bf16x4 d2[4];
#pragma unroll
    for (int o = 0; o < 4; ++o) {
      f32x4 d;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        g3[o][i] += h2[o][i] * dy;
        d[i] = h2[o][i] > 0.f ? dy * nr.w3[o][i] : 0.f;
        gb2[o][i] += d[i];
      }
      d2[o] = to_bf16x4(d);
    }
    // dH1 = W2 dH2 where H1 > 0; db1 = dH1
    bf16x4 d1[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      f32x4 acc = zero;
#pragma unroll
      for (int k = 0; k < 4; ++k) acc = mfma16(w2b[t][k], d2[k], acc);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[i] = h1[t][i] > 0 ? acc[i] : 0.f;  // H1 is not negative: its bits say whether it is 0
        gb1[t][i] += acc[i];
      }
      d1[t] = to_bf16x4(acc);
    }
    __syncthreads();  // the previous rows are no longer read
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int u = 16 * t + 4 * g4 + i;
        H1[u][col] = (uint16_t)h1[t][i];
        D2[u][col] = (uint16_t)d2[t][i];
        D1[u][col] = (uint16_t)d1[t][i];
      }
#pragma unroll
    for (int i = 0; i < 4; ++i) XT[4 * g4 + i][col] = (uint16_t)x[i];
    __syncthreads();
    // dW2 = H1^T dH2 and dW1 = X^T dH1 over the 64 rows, 32 per MFMA
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int k0 = 32 * m + 8 * g4;
      auto frag = [&](const uint16_t (*a)[LD], int u) {
        return *reinterpret_cast<const bf16x8 *>(&a[u][k0]);
      };
      const bf16x8 a = frag(H1, 16 * w + l16);
#pragma unroll
      for (int c = 0; c < 4; ++c)
        gw2[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, frag(D2, 16 * c + l16), gw2[c], 0, 0, 0);
      gw1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(XT, l16), frag(D1, 16 * w + l16), gw1, 0, 0, 0);
    }
  }
  float *p = part + (size_t)blockIdx.x * kGradStride;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 4 * g4 + i;
#pragma unroll
    for (int c = 0; c < 4; ++c) p[OW2 + (16 * w + r) * NH + 16 * c + l16] = gw2[c][i];
    if (r < NIN) p[OW1 + r * NH + 16 * w + l16] = gw1[i];
  }
  // per-unit sums: over the wave's 16 rows, then over the 4 waves
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float a = row_sum(g3[t][i]), b = row_sum(gb2[t][i]), c = row_sum(gb1[t][i]);
      if (l16 == 15) {
        const int u = 16 * t + 4 * g4 + i;
        red[0][w][u] = a;
        red[1][w][u] = b;
        red[2][w][u] = c;
      }
    }
  sq = row_sum(sq);
  sdy = row_sum(sdy);
  if (lane == 15) {
    red2[0][w] = sq;
    red2[1][w] = sdy;
  }
  __syncthreads();
  if (w < 3) {
    const float v = (red[w][0][lane] + red[w][1][lane]) + (red[w][2][lane] + red[w][3][lane]);
    p[(w == 0 ? OW3 : w == 1 ? OB2 : OB1) + lane] = v;
  } else if (lane < 2) {
    const float v = (red2[lane][0] + red2[lane][1]) + (red2[lane][2] + red2[lane][3]);
    p[lane == 0 ? NPARAM : OB3] = v;
  }
}

// Forward only over given rows (tests, scoring): a wave takes 64 rows.
__global__ void __launch_bounds__(256)
k_mlp_forward(const MlpDev *__restrict__ net, const float *__restrict__ Xg, int n,
              float *__restrict__ y) {
  const int lane = threadIdx.x & 63, l16 = lane & 15;
  const long row0 = ((long)blockIdx.x * 4 + (threadIdx.x >> 6)) * 64;
  if (row0 >= n) return;  // the whole wave
  const NetRegs nr(net);
  float v = 0.f;
#pragma unroll
  for (int R = 0; R < 4; ++R) {
    const long row = row0 + 16 * R + l16;
    bf16x4 h1[4];
    f32x4 h2[4];
    const float t = forward_tile(nr, load_x(Xg, row, row < n), h1, h2);
    if ((lane >> 4) == R) v = t;  // lane 16 R + l16 keeps row 16 R + l16
  }
  if (row0 + lane < n) y[row0 + lane] = v;
}

// Gradient of parameter p (and, at p = NPARAM, the sum of squared errors,
// added to *loss) from the nb workgroups' sums, in a fixed order: 4 strided
// partial sums per parameter, then those.  ADAM: the FP32 master parameters
// take the step and the kernels' copies are stored; otherwise the gradient
// goes to G.
template <bool ADAM>
__global__ void __launch_bounds__(256)
k_reduce_grad(const float *__restrict__ part, int nb, float *__restrict__ P, float *__restrict__ G,
              float *__restrict__ m1, float *__restrict__ m2, float lr, float b1, float b2,
              float eps, float c1, float c2, MlpDev *__restrict__ net, float *__restrict__ loss) {
  __shared__ float s[4][64];
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + lane;
  const int ic = i <= NPARAM ? i : NPARAM;
  float g = 0.f;
#pragma unroll 8
  for (int b = q; b < nb; b += 4) g += part[(size_t)b * kGradStride + ic];
  s[q][lane] = g;
  __syncthreads();
  if (q != 0 || i > NPARAM) return;
  g = (s[0][lane] + s[1][lane]) + (s[2][lane] + s[3][lane]);
  if (i == NPARAM) {
    *loss += g;
    return;
  }
  if constexpr (ADAM) {
    const float a = b1 * m1[i] + (1.f - b1) * g;
    const float v = b2 * m2[i] + (1.f - b2) * g * g;
    m1[i] = a;
    m2[i] = v;
    const float w = P[i] - lr * (a / c1) / (sqrtf(v / c2) + eps);
    P[i] = w;
    put_param(net, i, w);
  } else {
    G[i] = g;
  }
}

__global__ void k_pack_net(const float *__restrict__ P, MlpDev *__restrict__ net) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < NPARAM) put_param(net, i, P[i]);
}

// ---- descriptors -------------------------------------------------------------
// A sphere's position, one aligned record: a wave's lanes read 64 spheres, and
// two loads of it occupy the compute unit's address path two thirds as long as
// three of an array each (scores of 50260 free voxels 51 -> 39 us, 2^20 sorted
// training rows at N = 4000 648 -> 566).
struct __attribute__((aligned(32))) Pos {
  double x, y, z, pad;
};

struct NGrid {  // CSR observable grid (side >= 1.5) over one replica
  int nx, ny, nz;
  double sx, sy, sz, ix, iy, iz, lx, ly, lz;  // ix = 1.0 / sx ...
  const int *start;
  const Pos *p;
};

// Candidate range of one row (dx, dy) of the 27-cell stencil: the row's z
// cells hold consecutive entries of the CSR arrays, so the row is one range
// [a0, a1), plus a second [b0, b1) where the stencil wraps around z (the
// cell at the far end).  With fewer than 3 cells along z the row is every
// cell, once.
__device__ __forceinline__ void row_ranges(const NGrid &g, int base, int cz, int &a0, int &a1,
                                           int &b0, int &b1) {
  int ac0, ac1, bc0 = 0, bc1 = 0;  // cell index ranges [ac0, ac1), [bc0, bc1) within the row
  if (g.nz >= 3) {
    if (cz == 0) {
      ac0 = 0, ac1 = 2, bc0 = g.nz - 1, bc1 = g.nz;
    } else if (cz == g.nz - 1) {
      ac0 = g.nz - 2, ac1 = g.nz, bc0 = 0, bc1 = 1;
    } else {
      ac0 = cz - 1, ac1 = cz + 2;
    }
  } else {
    ac0 = 0, ac1 = g.nz;
  }
  // four loads with no branch around them (an empty second range reads one
  // entry twice), so the rows' loads all issue before any is waited for
  a0 = g.start[base + ac0];
  a1 = g.start[base + ac1];
  b0 = g.start[base + bc0];
  b1 = g.start[base + bc1];
}

// f(squared distance) of every sphere in the 27 cells around q, row by row.
// A row's ranges are loaded while the row before it is scanned, and its
// spheres go CH at a time with their loads issued together (past the row's
// end a lane repeats its last sphere and f is not called).  One loop body
// for all rows: with the 9 rows unrolled the search was 90 KB of code, several
// times the instruction cache, read once by each wave (scores of 50260 free
// voxels 64 -> 50 us, with the network's layers in registers).
template <int CH, class F>
__device__ __forceinline__ void scan_rows(const NGrid &g, double qx, double qy, double qz, F &&f) {
  const int cx = search_cell(qx, g.ix, g.nx), cy = search_cell(qy, g.iy, g.ny),
            cz = search_cell(qz, g.iz, g.nz);
  auto load = [&](int r, int &a0, int &a1, int &b0, int &b1) {
    const int dx = r / 3 - 1, dy = r % 3 - 1;
    const bool ok = stencil_axis_ok(dx, g.nx) && stencil_axis_ok(dy, g.ny);
    const int base = ok ? (wrap_index(cx + dx, g.nx) * g.ny + wrap_index(cy + dy, g.ny)) * g.nz : 0;
    row_ranges(g, base, cz, a0, a1, b0, b1);
    if (!ok) a1 = a0, b1 = b0;  // a row the stencil leaves out
  };
  int a0, a1, b0, b1;
  load(0, a0, a1, b0, b1);
#pragma unroll 1
  for (int r = 0; r < 9; ++r) {
    const int la = a1 - a0, len = la + (b1 - b0), pa = a0, pb = b0 - la;
    if (r < 8) load(r + 1, a0, a1, b0, b1);
#pragma unroll 1
    for (int u0 = 0; u0 < len; u0 += CH) {
      double ox[CH], oy[CH], oz[CH];
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        const int e = min(u0 + u, len - 1);
        const int q = e + (e < la ? pa : pb);
        const Pos &o = g.p[q];
        ox[u] = o.x;
        oy[u] = o.y;
        oz[u] = o.z;
      }
#pragma unroll
      for (int u = 0; u < CH; ++u)
        if (u0 + u < len) f(dist2(qx, qy, qz, ox[u], oy[u], oz[u], g.lx, g.ly, g.lz));
    }
  }
}

// 12 smallest squared distances (ascending) from q to sphere centres in the
// 27 cells around q; entries not found stay at `far2`.  The result depends
// only on the set of candidates, not on the order they are met.  A new
// distance d enters the sorted list as best[k] = median(best[k-1], best[k], d).
__device__ __forceinline__ void take12(float d, float best[NIN]) {
#pragma unroll
  for (int k = NIN - 1; k > 0; --k) best[k] = __builtin_amdgcn_fmed3f(best[k - 1], best[k], d);
  best[0] = fminf(best[0], d);
}

__device__ __forceinline__ void nearest12(const NGrid &g, double qx, double qy, double qz,
                                          float far2, float best[NIN]) {
#pragma unroll
  for (int k = 0; k < NIN; ++k) best[k] = far2;
  scan_rows<8>(g, qx, qy, qz, [&](double d2) { take12((float)d2, best); });
}

// The smallest of those alone.  A rounded minimum is the minimum of the
// rounded distances, so it is nearest12's best[0].
__device__ __forceinline__ float nearest1(const NGrid &g, double qx, double qy, double qz,
                                          float far2) {
  double m = (double)far2;
  scan_rows<8>(g, qx, qy, qz, [&](double d2) { m = fmin(m, d2); });
  return (float)m;
}

struct Vox {
  int mx, my, mz;
  double vx, vy, vz;  // voxel edges
  long V;
};

__device__ __forceinline__ void voxel_centre(const Vox &vx, long v, double &x, double &y,
                                             double &z) {
  const int iz = (int)(v % vx.mz);
  const long t = v / vx.mz;
  const int iy = (int)(t % vx.my), ix = (int)(t / vx.my);
  x = (ix + 0.5) * vx.vx;
  y = (iy + 0.5) * vx.vy;
  z = (iz + 0.5) * vx.vz;
}

// descriptor entries: distances minus one diameter
__device__ __forceinline__ void descriptor(const NGrid &g, double x, double y, double z,
                                           float far2, float out[NIN]) {
  float best[NIN];
  nearest12(g, x, y, z, far2, best);
#pragma unroll
  for (int k = 0; k < NIN; ++k) out[k] = sqrtf(best[k]) - 1.0f;
}

__global__ void __launch_bounds__(256)
k_point_descriptors(NGrid g, const double *__restrict__ q, int m, float far2,
                    float *__restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  float d[NIN];
  descriptor(g, q[3 * i], q[3 * i + 1], q[3 * i + 2], far2, d);
  for (int k = 0; k < NIN; ++k) out[(size_t)i * NIN + k] = d[k];
}

__device__ __forceinline__ int cell_of(const NGrid &g, double x, double y, double z) {
  return (search_cell(x, g.ix, g.nx) * g.ny + search_cell(y, g.iy, g.ny)) * g.nz + search_cell(z, g.iz, g.nz);
}

// Uniform point i of Philox stream (key, sample), and the centre of the voxel
// that holds it.
struct TrainingPoints {
  uint32_t k0, k1;
  unsigned long long sample;
  __device__ __forceinline__ void operator()(const NGrid &g, const Vox &vx, long long i, double q[3],
                                             double c[3]) const {
    uint32_t u[4];
    philox4x32_10((uint32_t)i, (uint32_t)((unsigned long long)i >> 32), (uint32_t)sample,
                  0x57490000u | (uint32_t)((sample >> 32) & 0xFFFFu), k0, k1, u);
    q[0] = u32_unit_closed(u[0]) * g.lx;
    q[1] = u32_unit_closed(u[1]) * g.ly;
    q[2] = u32_unit_closed(u[2]) * g.lz;
    int ix = (int)(q[0] / vx.vx), iy = (int)(q[1] / vx.vy), iz = (int)(q[2] / vx.vz);
    ix = min(ix, vx.mx - 1);
    iy = min(iy, vx.my - 1);
    iz = min(iz, vx.mz - 1);
    const long v = ((long)ix * vx.my + iy) * vx.mz + iz;
    voxel_centre(vx, v, c[0], c[1], c[2]);
  }
};

// Points are worked on in the order of their voxels' cells, so that a wave
// reads the spheres of one or two cells instead of 64 cells' (each of these
// scattered lines takes the compute unit's address path a cycle, which
// bounded the rows).  The rows stay where they were: only which lane makes
// which row changes.  rank[i] = place of point i among its cell's; cnt = the
// cells' counts.  Up to kLdsCells cells a workgroup counts its points in LDS
// first: on a grid of few cells its one addition a cell takes the place of
// hundreds to the same few words.
constexpr int kLdsCells = 8192;
constexpr int kSortThreads = 1024;

template <bool LDS>
__global__ void __launch_bounds__(kSortThreads)
k_training_count(NGrid g, Vox vx, TrainingPoints point, long long first, int n, int *__restrict__ cnt,
                 int *__restrict__ rank) {
  __shared__ int own[LDS ? kLdsCells : 1];
  const int i = blockIdx.x * kSortThreads + threadIdx.x;
  const int C = g.nx * g.ny * g.nz;
  if constexpr (LDS) {
    for (int c = threadIdx.x; c < C; c += kSortThreads) own[c] = 0;
    __syncthreads();
  }
  int cell = 0, r = 0;
  if (i < n) {
    double q[3], c[3];
    point(g, vx, first + i, q, c);
    cell = cell_of(g, c[0], c[1], c[2]);
    r = atomicAdd(LDS ? &own[cell] : &cnt[cell], 1);
  }
  if constexpr (LDS) {
    __syncthreads();
    for (int c = threadIdx.x; c < C; c += kSortThreads) {
      const int k = own[c];
      if (k) own[c] = atomicAdd(&cnt[c], k);
    }
    __syncthreads();
    r += own[cell];
  }
  if (i < n) rank[i] = r;
}

__global__ void __launch_bounds__(256)
k_training_order(NGrid g, Vox vx, TrainingPoints point, long long first, int n,
                 const int *__restrict__ start, const int *__restrict__ rank, int *__restrict__ order) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double q[3], c[3];
  point(g, vx, first + i, q, c);
  order[start[cell_of(g, c[0], c[1], c[2])] + rank[i]] = i;
}

// Training rows of points first .. first + n - 1, in the given order (any
// without one): input = descriptor of the voxel holding the point, target
// = -beta * max(0, 1 - d).
__global__ void __launch_bounds__(256)
k_training_rows(NGrid g, Vox vx, TrainingPoints point, long long first, long long n,
                const int *__restrict__ order, float far2, float beta, float *__restrict__ X,
                float *__restrict__ T) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const long long i = first + (order ? order[t] : t);
  double q[3], c[3];
  point(g, vx, i, q, c);
  const float dmin = sqrtf(nearest1(g, q[0], q[1], q[2], far2));
  T[i] = -beta * fmaxf(0.f, 1.f - dmin);
  float d[NIN];
  descriptor(g, c[0], c[1], c[2], far2, d);
  for (int k = 0; k < NIN; ++k) X[(size_t)i * NIN + k] = d[k];
}

// Network scores of a block's 256 voxels from their descriptors (one wave per
// 64 voxels, MFMA) and the block's max and sum exp(f - max).
__device__ void score_block(const MlpDev *__restrict__ net, uint16_t (*X)[64 * KIN], float *red,
                            const float d[NIN], bool ok, long v, float *__restrict__ f,
                            float *__restrict__ bmax, float *__restrict__ bsum) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, g4 = lane >> 4;
#pragma unroll
  for (int k = 0; k < KIN; k += 4) {
    f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (k + i < NIN) c[i] = d[k + i];
    *reinterpret_cast<bf16x4 *>(&X[w][lane * KIN + k]) = to_bf16x4(c);
  }
  wave_lds_sync();
  float val = 0.f;
  {
    const NetRegs nr(net);
#pragma unroll
    for (int R = 0; R < 4; ++R) {
      bf16x4 h1[4];
      f32x4 h2[4];
      const float t = forward_tile(
          nr, *reinterpret_cast<const bf16x4 *>(&X[w][(R * 16 + l16) * KIN + 4 * g4]), h1, h2);
      if (g4 == R) val = t;  // lane 16 R + l16 keeps row 16 R + l16
    }
  }
  if (ok) f[v] = val;
  float m = ok ? val : -INFINITY;
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if (lane == 0) red[w] = m;
  __syncthreads();
  const float bm = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float e = ok ? expf(val - bm) : 0.f;
  for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o, 64);
  __syncthreads();
  if (lane == 0) red[4 + w] = e;
  __syncthreads();
  if (threadIdx.x == 0) {
    bmax[blockIdx.x] = bm;
    bsum[blockIdx.x] = red[4] + red[5] + red[6] + red[7];
  }
}

// Scores of all voxels: descriptor + network, fused (descriptors never leave
// the chip).  Block = 256 consecutive voxels, each searching the grid alone.
__global__ void __launch_bounds__(256)
k_voxel_scores(NGrid g, Vox vx, float far2, const MlpDev *__restrict__ net,
               float *__restrict__ f, float *__restrict__ bmax, float *__restrict__ bsum) {
  __shared__ __attribute__((aligned(16))) uint16_t X[4][64 * KIN];
  __shared__ float red[8];
  const long v = (long)blockIdx.x * 256 + threadIdx.x;
  float d[NIN];
  if (v < vx.V) {
    double cx, cy, cz;
    voxel_centre(vx, v, cx, cy, cz);
    descriptor(g, cx, cy, cz, far2, d);
  } else {
    for (int k = 0; k < NIN; ++k) d[k] = 0.f;
  }
  score_block(net, X, red, d, v < vx.V, v, f, bmax, bsum);
}

// The same over 4 x 8 x 8 voxel tiles (one wave per x layer): the block first
// gathers into LDS, as FP32 offsets from the tile centre, every sphere whose
// minimum-image offset lies within the tile's half extent + smin on each
// axis (a superset of the spheres within smin of any of its voxel centres),
// then each voxel takes its 12 nearest from LDS.  The host uses it only when
// every box edge exceeds 2 (tile extent + smin), so one image serves the
// whole tile.  A tile whose set would overflow the LDS list (impossible
// below close packing: a 4 x 5 x 5 sigma^3 box holds at most ~254 spheres)
// searches the grid per voxel instead.
constexpr int TX = 4, TY = 8, TZ = 8, TCAP = 320;

__global__ void __launch_bounds__(256)
k_voxel_scores_tiled(NGrid g, Vox vx, float far2, double smin, const MlpDev *__restrict__ net,
                     float *__restrict__ f, float *__restrict__ bmax, float *__restrict__ bsum) {
  __shared__ __attribute__((aligned(16))) uint16_t X[4][64 * KIN];
  __shared__ float red[8];
  __shared__ float qx[TCAP], qy[TCAP], qz[TCAP];
  __shared__ int ncand;
  if (threadIdx.x == 0) ncand = 0;
  __syncthreads();
  const int ntz = (vx.mz + TZ - 1) / TZ, nty = (vx.my + TY - 1) / TY;
  const int bz = blockIdx.x % ntz, by = (blockIdx.x / ntz) % nty, bx = blockIdx.x / (ntz * nty);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int ix = bx * TX + w, iy = by * TY + (lane >> 3), iz = bz * TZ + (lane & 7);
  const bool ok = ix < vx.mx && iy < vx.my && iz < vx.mz;
  // tile centre and the half extent of the gathered box
  const double ccx = (bx * TX + TX * 0.5) * vx.vx, ccy = (by * TY + TY * 0.5) * vx.vy,
               ccz = (bz * TZ + TZ * 0.5) * vx.vz;
  const double ex = (TX - 1) * 0.5 * vx.vx + smin, ey = (TY - 1) * 0.5 * vx.vy + smin,
               ez = (TZ - 1) * 0.5 * vx.vz + smin;
  // grid cells overlapping the box, per axis (all cells when it spans them)
  int lo[3], nc[3];
  const double cc[3] = {ccx, ccy, ccz}, ee[3] = {ex, ey, ez}, side[3] = {g.sx, g.sy, g.sz};
  const int gn[3] = {g.nx, g.ny, g.nz};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int l = (int)floor((cc[a] - ee[a]) / side[a]);
    const int h = (int)floor((cc[a] + ee[a]) / side[a]);
    nc[a] = h - l + 1;
    lo[a] = l;
    if (nc[a] >= gn[a]) {
      nc[a] = gn[a];
      lo[a] = 0;
    }
  }
  const int ncell = nc[0] * nc[1] * nc[2];
  for (int k = threadIdx.x; k < ncell; k += blockDim.x) {
    const int kx = k / (nc[1] * nc[2]), ky = (k / nc[2]) % nc[1], kz = k % nc[2];
    const int c = (wrap_index(lo[0] + kx, g.nx) * g.ny + wrap_index(lo[1] + ky, g.ny)) * g.nz +
                  wrap_index(lo[2] + kz, g.nz);
    for (int p = g.start[c]; p < g.start[c + 1]; ++p) {
      const double dx = min_image(g.p[p].x - ccx, g.lx, g.lx / 2.0);
      const double dy = min_image(g.p[p].y - ccy, g.ly, g.ly / 2.0);
      const double dz = min_image(g.p[p].z - ccz, g.lz, g.lz / 2.0);
      if (fabs(dx) <= ex && fabs(dy) <= ey && fabs(dz) <= ez) {
        const int slot = atomicAdd(&ncand, 1);
        if (slot < TCAP) {
          qx[slot] = (float)dx;
          qy[slot] = (float)dy;
          qz[slot] = (float)dz;
        }
      }
    }
  }
  __syncthreads();
  const int n = ncand;
  float d[NIN];
  if (ok) {
    const double vxc = (ix + 0.5) * vx.vx, vyc = (iy + 0.5) * vx.vy, vzc = (iz + 0.5) * vx.vz;
    if (n <= TCAP) {
      float best[NIN];
#pragma unroll
      for (int k = 0; k < NIN; ++k) best[k] = far2;
      const float ox = (float)(vxc - ccx), oy = (float)(vyc - ccy), oz = (float)(vzc - ccz);
      for (int q = 0; q < n; ++q) {
        const float ax = qx[q] - ox, ay = qy[q] - oy, az = qz[q] - oz;
        const float d2 = ax * ax + ay * ay + az * az;
        take12(d2, best);
      }
#pragma unroll
      for (int k = 0; k < NIN; ++k) d[k] = sqrtf(best[k]) - 1.0f;
    } else {
      descriptor(g, vxc, vyc, vzc, far2, d);
    }
  } else {
    for (int k = 0; k < NIN; ++k) d[k] = 0.f;
  }
  const long v = ((long)ix * vx.my + iy) * vx.mz + iz;
  score_block(net, X, red, d, ok, v, f, bmax, bsum);
}

// Voxels that can hold a free point.  Every point of a voxel lies within
// half its diagonal h of the voxel's centre, so a voxel whose centre is
// closer than r = 1 - h to a sphere centre lies inside that sphere's
// exclusion zone and no insertion in it can succeed.  The proposal gives such
// voxels no network mass (q_v = (1 - mix) / V, the uniform part alone, still
// > 0, so the estimate stays unbiased; their score reads -inf in
// hsmc_gpu_proposal_scores) and the network scores only the others.
//
// Two passes.  k_mark_blocked: one wave per sphere marks (a byte flag)
// every voxel whose centre's squared distance to it, in FP64 as
// compute_dist evaluates it (minimum image), is below r^2 -- so a voxel is
// marked exactly when some sphere blocks it; all marks store the same 1.
// k_free_tiles: one wave per tile of 4 x 8 x 8 voxels puts the unmarked
// ("free") voxels in the tile's own range of `slots` (256 per tile, in the
// tile's x, y, z order) with their number in cnt[tile]; k_gather_free packs
// them into one list (tile order, then that order) for k_voxel_scores_list.
// No global atomics: the tile counts are prefix-summed instead.  Scores are
// written for free voxels only; the flags tell the others apart.
struct Box3 {
  double lx, ly, lz;
  double ux, uy, uz;  // voxels per unit length
};

// First candidate voxel index for centres (i + 0.5) * v within r of p: the
// centres within r have i in the open interval (x, x + 2r/v) with
// x = (p - r)/v - 0.5, and the 8 indices from floor(x - 1e-9) cover it when
// 2r/v + 1 < 8 - 1e-6 (the host checks; 6.27 for voxels of edge 0.25), also
// where rounding, of 1/v too, puts x on the other side of an integer.  The
// distance test then decides each candidate.  (Three divisions a sphere were
// a third of the kernel's instructions, which bound it: 42 us for N = 108000.)
__device__ __forceinline__ int voxel_first(double p, double r, double per_unit) {
  return (int)floor((p - r) * per_unit - 0.5 - 1e-9);
}

__device__ __forceinline__ int wrap_voxel(int i, int m) {
  return i < 0 ? i + m : (i >= m ? i - m : i);
}

// Lane t's value of v, read into every lane (t the same in all of them).
__device__ __forceinline__ double lane_value(double v, int t) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, t);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), t);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__global__ void __launch_bounds__(256)
k_mark_blocked(const double *__restrict__ x, const double *__restrict__ y,
               const double *__restrict__ z, int N, Vox vx, Box3 b, double r,
               unsigned char *__restrict__ flag) {
  const int lane = threadIdx.x & 63;
  const int p = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (p >= N) return;  // the whole wave
  const double px = x[p], py = y[p], pz = z[p];
  const int lx = voxel_first(px, r, b.ux), ly = voxel_first(py, r, b.uy), lz = voxel_first(pz, r, b.uz);
  const double r2 = r * r;
  // 8 x 8 x 8 candidates: lane's (y, z) column, 8 x-layers.  The squared
  // distance is compute_dist's (dx^2 + dy^2) + dz^2 with the minimum image
  // per axis.  Its x part is the same in every lane, so lane k < 8 computes
  // layer k's index and dx^2 once and each layer reads them from that lane.
  const int kx = lane & 7;
  const int ixk = wrap_voxel(lx + kx, vx.mx);
  const double dxk = image_mag((ixk + 0.5) * vx.vx - px, b.lx);
  const double dx2k = (unsigned)ixk < (unsigned)vx.mx ? dxk * dxk : INFINITY;
  const int iy = wrap_voxel(ly + (lane >> 3), vx.my), iz = wrap_voxel(lz + (lane & 7), vx.mz);
  const double dy = image_mag((iy + 0.5) * vx.vy - py, b.ly);
  const double dz = image_mag((iz + 0.5) * vx.vz - pz, b.lz);
  // (a sphere outside the box has candidates off the voxels: none of them)
  const double dy2 = (unsigned)iy < (unsigned)vx.my ? dy * dy : INFINITY,
               dz2 = (unsigned)iz < (unsigned)vx.mz ? dz * dz : INFINITY;
  const long col = (long)iy * vx.mz + iz, layer = (long)vx.my * vx.mz;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const double dx2 = lane_value(dx2k, k);
    const int ix = __builtin_amdgcn_readlane(ixk, k);
    if (dx2 + dy2 + dz2 < r2) flag[(long)ix * layer + col] = 1;
  }
}

__global__ void __launch_bounds__(256)
k_free_tiles(Vox vx, const unsigned char *__restrict__ flag, int *__restrict__ slots,
             int *__restrict__ cnt, long tiles) {
  const long tile = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tile >= tiles) return;  // the whole wave
  const int ntz = (vx.mz + TZ - 1) / TZ, nty = (vx.my + TY - 1) / TY;
  const int bz = (int)(tile % ntz), by = (int)((tile / ntz) % nty), bx = (int)(tile / ((long)ntz * nty));
  // lane l: row (x = l / 16, y = (l / 2) % 8) of the tile, voxels z = 4 (l % 2) .. + 3,
  // so lane order then z is the tile's x, y, z order
  const int lane = threadIdx.x & 63;
  const int ix = bx * TX + (lane >> 4), iy = by * TY + ((lane >> 1) & 7), iz0 = bz * TZ + 4 * (lane & 1);
  const bool row = ix < vx.mx && iy < vx.my;
  const long v0 = ((long)ix * vx.my + iy) * vx.mz + iz0;
  unsigned char f[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) f[k] = flag[row && iz0 + k < vx.mz ? v0 + k : 0];  // no branch around the loads
  int bits = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) bits |= (row && iz0 + k < vx.mz && f[k] == 0) ? 1 << k : 0;
  const int n = __popc(bits);
  const int incl = group_inclusive_sum<64>(n);
  int *out = slots + (size_t)tile * 256 + (incl - n);
#pragma unroll
  for (int k = 0, j = 0; k < 4; ++k)
    if ((bits >> k) & 1) out[j++] = (int)(v0 + k);
  if (lane == 63) cnt[tile] = incl;
}

// Pack the tiles' free voxels into one list: tile t's cnt[t] entries go to
// list[off[t] ...] (off: exclusive prefix sum of cnt); one wave per tile.  The
// number of free voxels goes to the host.
__global__ void __launch_bounds__(256)
k_gather_free(const int *__restrict__ slots, const int *__restrict__ cnt,
              const int *__restrict__ off, int *__restrict__ list, long tiles,
              unsigned long long *__restrict__ host) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *host = (unsigned long long)off[tiles];
  const long t = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= tiles) return;
  const int n = cnt[t], o = off[t];
  for (int k = threadIdx.x & 63; k < n; k += 64) list[o + k] = slots[(size_t)t * 256 + k];
}

// Network scores of the free voxels list[0..n) (descriptor + network, as
// k_voxel_scores does for every voxel), and per block the max and sum of
// exp(f - max) over them.
__global__ void __launch_bounds__(256)
k_voxel_scores_list(NGrid g, Vox vx, float far2, const MlpDev *__restrict__ net,
                    const int *__restrict__ list, int n, float *__restrict__ f,
                    float *__restrict__ bmax, float *__restrict__ bsum) {
  __shared__ __attribute__((aligned(16))) uint16_t X[4][64 * KIN];
  __shared__ float red[8];
  const int i = blockIdx.x * 256 + threadIdx.x;
  const bool ok = i < n;
  const long v = ok ? (long)list[i] : 0;
  float d[NIN];
  if (ok) {
    double cx, cy, cz;
    voxel_centre(vx, v, cx, cy, cz);
    descriptor(g, cx, cy, cz, far2, d);
  } else {
    for (int k = 0; k < NIN; ++k) d[k] = 0.f;
  }
  score_block(net, X, red, d, ok, v, f, bmax, bsum);
}

// Network part of the proposal mass of a free voxel v:
// mix * softmax(f)_v = mix * exp(f_v - fmax) / sumexp, with st[0] = fmax and
// st[1] = sumexp (on the device, written by k_cdf_local).
__device__ __forceinline__ double network_mass(const float *__restrict__ f, long v,
                                               const double *__restrict__ st, double mix) {
  return mix * exp((double)f[v] - st[0]) / st[1];
}

// st[0] = max of the blocks' maxima, st[1] = sum of their sums of
// exp(f - max) rescaled to st[0], each in a fixed order (256 strided
// partials, then a tree), for the whole workgroup (at least 256 threads).
__device__ __forceinline__ void softmax_stats(const float *__restrict__ bmax,
                                              const float *__restrict__ bsum, long nb, double st[2]) {
  __shared__ double s[256];
  const int t = threadIdx.x;
  double m = -INFINITY;
  if (t < 256) {
    for (long b = t; b < nb; b += 256) m = fmax(m, (double)bmax[b]);
    s[t] = m;
  }
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w) s[t] = fmax(s[t], s[t + w]);
    __syncthreads();
  }
  const double fm = s[0];
  __syncthreads();
  if (t < 256) {
    double e = 0.0;
    for (long b = t; b < nb; b += 256) e += (double)bsum[b] * exp((double)bmax[b] - fm);
    s[t] = e;
  }
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w) s[t] += s[t + w];
    __syncthreads();
  }
  st[0] = fm;
  st[1] = s[0];
}

// The same by one workgroup, for a proposal of many free voxels.
__global__ void __launch_bounds__(256)
k_softmax_stats(const float *__restrict__ bmax, long nb, double *__restrict__ stats) {
  double st[2];
  softmax_stats(bmax, bmax + nb, nb, st);
  if (threadIdx.x == 0) {
    stats[0] = st[0];
    stats[1] = st[1];
    stats[2] = 0.0;
  }
}

// The statistics of a proposal with no free voxel (every voxel keeps the
// uniform part alone).
__global__ void k_empty_stats(double *__restrict__ st) {
  if (threadIdx.x == 0) {
    st[0] = 0.0;
    st[1] = 1.0;
    st[2] = 0.0;
  }
}

// Cumulative network mass over the free-voxel list (list order): inclusive
// sums within blocks of 4096 entries (+ block totals), then the blocks'
// exclusive offsets added, the total behind the block totals.  The offsets
// are a scan of the totals, of up to kScanWave of them by every workgroup of
// the adding kernel for itself, of more by a kernel in between (the same
// additions either way): with the totals, the hits and the number of free
// voxels also going to the host from the kernels that know them, one insertion
// call at N = 108000 takes 292 us, 342 with a kernel for each of these steps,
// two copies and two waits.  With bmax the softmax totals are taken from the
// scoring kernel's nparts block partials first (each workgroup for itself,
// the first stores them); otherwise st holds them already.
constexpr int kScanWave = 64;
// Up to here every workgroup of k_cdf_local takes the totals for itself, above
// one workgroup does before them: a call at N = 108000 with 4520 partials 483
// and 488 us, with 9985 664 and 647, with 58864 2163 and 1425, with 82004 4543
// and 2749 (the work of the first grows with the square of the free voxels).
constexpr long kStatsParts = 8192;

__global__ void __launch_bounds__(1024)
k_cdf_local(const float *__restrict__ f, const int *__restrict__ list, long V, const float *__restrict__ bmax,
            long nparts, double *__restrict__ stats, double mix, double *__restrict__ cdf,
            double *__restrict__ bsum) {
  __shared__ double s[2][1024];
  const long base = (long)blockIdx.x * 4096;
  double st[2];
  if (bmax) {
    softmax_stats(bmax, bmax + nparts, nparts, st);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      stats[0] = st[0];
      stats[1] = st[1];
      stats[2] = 0.0;
    }
  } else {
    st[0] = stats[0];
    st[1] = stats[1];
  }
  double v[4], tot = 0.0;
  for (int j = 0; j < 4; ++j) {
    const long i = base + threadIdx.x * 4 + j;
    v[j] = i < V ? network_mass(f, list[i], st, mix) : 0.0;
    tot += v[j];
  }
  // s[0] and s[1] in turn: one barrier a step
  double incl = tot;
  for (int d = 1, b = 0; d < 1024; d <<= 1, b ^= 1) {
    s[b][threadIdx.x] = incl;
    __syncthreads();
    incl += (int)threadIdx.x >= d ? s[b][threadIdx.x - d] : 0.0;
  }
  double run = incl - tot;
  for (int j = 0; j < 4; ++j) {
    const long i = base + threadIdx.x * 4 + j;
    run += v[j];
    if (i < V) cdf[i] = run;
  }
  if (threadIdx.x == 1023) bsum[blockIdx.x] = incl;
}

__global__ void __launch_bounds__(1024) k_cdf_blocks(double *__restrict__ b, int nb) {
  __shared__ double part[1024];
  const int t = threadIdx.x, per = (nb + 1023) / 1024, lo = t * per, hi = min(nb, lo + per);
  double sum = 0.0;
  for (int i = lo; i < hi; ++i) sum += b[i];
  part[t] = sum;
  __syncthreads();
  for (int d = 1; d < 1024; d <<= 1) {
    const double v = t >= d ? part[t - d] : 0.0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  double run = part[t] - sum;
  for (int i = lo; i < hi; ++i) {
    const double bi = b[i];
    b[i] = run;
    run += bi;
  }
  __syncthreads();
  if (t == 1023) b[nb] = part[1023];
}

// SCAN: b holds the nb <= kScanWave block totals, scanned here (k_cdf_blocks'
// additions: steps of 1, 2, 4, ... and the own total taken off again).
template <bool SCAN>
__global__ void __launch_bounds__(256)
k_cdf_add(double *__restrict__ cdf, long V, double *__restrict__ b, int nb, double *__restrict__ total) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  double off = 0.0;
  const int mine = (int)((long)blockIdx.x * blockDim.x / 4096);  // 4096 is a multiple of the workgroup's entries
  if constexpr (SCAN) {
    const int lane = threadIdx.x & 63;
    const double own = lane < nb ? b[lane] : 0.0;
    double incl = own;
    for (int d = 1; d < 64; d <<= 1) {
      const double v = __shfl_up(incl, d, 64);
      incl += lane >= d ? v : 0.0;
    }
    off = __shfl(incl - own, mine, 64);
    if (blockIdx.x == 0 && threadIdx.x == 63) *total = incl;
  } else {
    off = b[mine];
  }
  if (i < V) cdf[i] += off;
}

// No sphere centre closer than 1 to q in the 27 cells around it (the
// overlap grid's cells are at least 1 wide).  The answer does not depend
// on the order of the cells, so they are visited nearest first (own cell,
// then the 6 sharing a face, with their ranges loaded together, then the
// rest): almost every proposed point overlaps a sphere, and usually one of
// those.
__device__ __forceinline__ bool widom_free(const NGrid &g1, double qx, double qy, double qz) {
  const int cx = search_cell(qx, g1.ix, g1.nx), cy = search_cell(qy, g1.iy, g1.ny),
            cz = search_cell(qz, g1.iz, g1.nz);
  auto cell_of = [&](int j, bool &ok) {
    int dx, dy, dz;
    stencil_by_distance(j, dx, dy, dz);
    ok = stencil_axis_ok(dx, g1.nx) && stencil_axis_ok(dy, g1.ny) && stencil_axis_ok(dz, g1.nz);
    return ok ? (wrap_index(cx + dx, g1.nx) * g1.ny + wrap_index(cy + dy, g1.ny)) * g1.nz +
                    wrap_index(cz + dz, g1.nz)
              : 0;
  };
  auto hit = [&](int b, int e) {
    for (int p = b; p < e; ++p)
      if (dist2(qx, qy, qz, g1.p[p].x, g1.p[p].y, g1.p[p].z, g1.lx, g1.ly, g1.lz) < 1.0)
        return true;
    return false;
  };
  int c7[7], b7[7], e7[7];
  bool ok7[7];
#pragma unroll
  for (int j = 0; j < 7; ++j) c7[j] = cell_of(j, ok7[j]);
#pragma unroll
  for (int j = 0; j < 7; ++j) b7[j] = g1.start[c7[j]];
#pragma unroll
  for (int j = 0; j < 7; ++j) e7[j] = g1.start[c7[j] + 1];
#pragma unroll
  for (int j = 0; j < 7; ++j)
    if (!ok7[j]) e7[j] = b7[j];
#pragma unroll
  for (int j = 0; j < 7; ++j)
    if (hit(b7[j], e7[j])) return false;
  for (int j = 7; j < 27; ++j) {
    bool ok;
    const int c = cell_of(j, ok);
    if (ok && hit(g1.start[c], g1.start[c + 1])) return false;
  }
  return true;
}

// Systematic sampling of n insertions from the proposal q_v = (1 - mix) / V
// + mix softmax(f)_v (the network part on free voxels only).  Insertion i
// takes t = (i + u0) / n * T, T = (1 - mix) + *total (the network mass
// summed over the free list, mix up to rounding; 0 with no free voxel).  t below 1 - mix
// falls in the uniform part, voxel floor(t V / (1 - mix)); above, in the
// network part: the free voxel whose cumulative-mass interval holds
// t - (1 - mix).  Each voxel thus covers (1 - mix) / V + its network mass
// of the t axis and gets floor or ceil of n q_v insertions, n q_v on
// average.  A point is uniform inside its voxel and, on a hit, weighs
// 1 / (V n q_v) with q_v its whole mass over T (the flags tell free voxels
// from blocked ones, whose network mass is 0).
__global__ void __launch_bounds__(256)
k_insert(NGrid g1, Vox vx, const double *__restrict__ cdf, const int *__restrict__ list,
         long nlist, const double *__restrict__ total, long n, double u0,
         const float *__restrict__ f, const unsigned char *__restrict__ flag,
         const double *__restrict__ st, double mix, uint32_t k0, uint32_t k1,
         unsigned long long sample, double *__restrict__ part,
         unsigned int *__restrict__ hits) {
  __shared__ double rs[4];
  __shared__ unsigned long long rh[4];
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const double un = 1.0 - mix, T = un + *total;
  double w = 0.0;
  unsigned long long h = 0;
  if (i < n) {
    const double t = ((double)i + u0) / (double)n * T;
    long v;
    if (t < un || nlist == 0) {
      v = (long)(t / un * (double)vx.V);
      if (v > vx.V - 1) v = vx.V - 1;
    } else {
      const double tn = t - un;
      long lo = 0, hi = nlist - 1;  // first free voxel whose cumulative mass exceeds tn
      while (lo < hi) {
        const long mid = (lo + hi) >> 1;
        if (cdf[mid] > tn)
          hi = mid;
        else
          lo = mid + 1;
      }
      v = list[lo];
    }
    const int iz = (int)(v % vx.mz);
    const long tv = v / vx.mz;
    const int iy = (int)(tv % vx.my), ix = (int)(tv / vx.my);
    uint32_t u[4];
    philox4x32_10((uint32_t)i, (uint32_t)(i >> 32), (uint32_t)sample,
                  0x4C490000u | (uint32_t)((sample >> 32) & 0xFFFFu), k0, k1, u);
    const double qx = (ix + ((double)u[0] + 0.5) * 0x1p-32) * vx.vx;
    const double qy = (iy + ((double)u[1] + 0.5) * 0x1p-32) * vx.vy;
    const double qz = (iz + ((double)u[2] + 0.5) * 0x1p-32) * vx.vz;
    if (widom_free(g1, qx, qy, qz)) {
      const double mass = un / (double)vx.V + (flag[v] == 0 ? network_mass(f, v, st, mix) : 0.0);
      w = 1.0 / ((double)vx.V * (double)n * (mass / T));
      h = 1;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    w += __shfl_xor(w, o, 64);
    h += __shfl_xor(h, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    rs[threadIdx.x >> 6] = w;
    rh[threadIdx.x >> 6] = h;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    // the block's weight and hits go to their own slots; the weights are summed
    // in a fixed order afterwards (k_sum_fixed), so an estimate never depends
    // on block timing
    part[blockIdx.x] = rs[0] + rs[1] + rs[2] + rs[3];
    hits[blockIdx.x] = (unsigned int)(rh[0] + rh[1] + rh[2] + rh[3]);
  }
}

// host[0] = sum of part[0..n), as bits, in an order fixed by n alone (256
// strided partial sums, then a pairwise tree), host[1] = sum of hits[0..n).
__global__ void __launch_bounds__(256) k_sum_fixed(const double *__restrict__ part,
                                                   const unsigned int *__restrict__ hits, long n,
                                                   unsigned long long *__restrict__ host) {
  __shared__ double s[256];
  __shared__ unsigned long long sh[256];
  double a = 0.0;
  unsigned long long h = 0;
#pragma unroll 4
  for (long i = threadIdx.x; i < n; i += 256) {
    a += part[i];
    h += hits[i];
  }
  s[threadIdx.x] = a;
  sh[threadIdx.x] = h;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      s[threadIdx.x] += s[threadIdx.x + w];
      sh[threadIdx.x] += sh[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    host[0] = (unsigned long long)__double_as_longlong(s[0]);
    host[1] = sh[0];
  }
}

// Build a CSR grid of one replica (side >= cut) into the given scratch slots.
int build_ngrid(hsmc_gpu_ctx *ctx, int replica, double cut, int slot0, NGrid &g);
int build_ngrid_pair(hsmc_gpu_ctx *ctx, int replica, double cut_a, double cut_b, NGrid &ga,
                     NGrid &gb);

}  // namespace

// ---- network object ----------------------------------------------------------
struct hsmc_gpu_mlp {
  hsmc_gpu_ctx *ctx = nullptr;
  float *P = nullptr, *G = nullptr, *m1 = nullptr, *m2 = nullptr;  // FP32 master, grad, Adam
  MlpDev *net = nullptr;
  float *loss = nullptr;
  long step = 0;
  // the proposal of the last configuration scored (replica, version, step,
  // voxel); its scores, flags, free list and softmax statistics stay in the
  // context's scratch
  int sc_replica = -1;
  unsigned long long sc_version = 0;
  long sc_step = -1;
  double sc_voxel = 0.0;
  double sc_mix = -1.0;   // mix of the cached cumulative network mass
  long sc_nfree = 0;      // free voxels of the cached proposal
  // the context's score stamp when this network last wrote the shared score
  // and cumulative-mass buffers; another writer (a second network, or
  // voxel_scores) changes the context's stamp and so invalidates the cache
  unsigned long long sc_stamp = 0;
};

namespace {

__global__ void k_grid_count2(const double *__restrict__ x, const double *__restrict__ y,
                              const double *__restrict__ z, int n, int nx, int ny, int nz,
                              double ix, double iy, double iz, int *__restrict__ cnt,
                              int *__restrict__ cellof) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int c = (search_cell(x[i], ix, nx) * ny + search_cell(y[i], iy, ny)) * nz + search_cell(z[i], iz, nz);
  cellof[i] = c;
  atomicAdd(&cnt[c], 1);
}

__global__ void k_grid_scatter2(const double *__restrict__ x, const double *__restrict__ y,
                                const double *__restrict__ z, int n, const int *__restrict__ cellof,
                                const int *__restrict__ start, int *__restrict__ fill,
                                Pos *__restrict__ p) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int c = cellof[i];
  const int pos = start[c] + atomicAdd(&fill[c], 1);
  p[pos] = Pos{x[i], y[i], z[i], 0.0};
}

// Two CSR grids of one replica filed in one pass: grid a's cells are the
// entries [0, Ca) of cnt and grid b's the entries [Ca, Ca + Cb), so one
// prefix sum over both gives grid a's starts in [0, n] and grid b's in
// [n, 2n], and both grids index one position array of 2n entries.
struct CellDims {
  int nx, ny, nz;
  double ix, iy, iz;  // reciprocal cell sides
};

__device__ __forceinline__ int cell_in(const CellDims &d, double x, double y, double z) {
  return (search_cell(x, d.ix, d.nx) * d.ny + search_cell(y, d.iy, d.ny)) * d.nz +
         search_cell(z, d.iz, d.nz);
}

__global__ void k_grid_count_pair(const double *__restrict__ x, const double *__restrict__ y,
                                  const double *__restrict__ z, int n, CellDims a, CellDims b,
                                  int ca, int *__restrict__ cnt, int4 *__restrict__ at) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double xi = x[i], yi = y[i], zi = z[i];
  const int c0 = cell_in(a, xi, yi, zi), c1 = ca + cell_in(b, xi, yi, zi);
  at[i] = make_int4(c0, c1, atomicAdd(&cnt[c0], 1), atomicAdd(&cnt[c1], 1));
}

__global__ void k_grid_scatter_pair(const double *__restrict__ x, const double *__restrict__ y,
                                    const double *__restrict__ z, int n,
                                    const int4 *__restrict__ at, const int *__restrict__ start,
                                    Pos *__restrict__ p) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double xi = x[i], yi = y[i], zi = z[i];
  const int4 a = at[i];
  const int p0 = start[a.x] + a.z, p1 = start[a.y] + a.w;
  p[p0] = p[p1] = Pos{xi, yi, zi, 0.0};
}

int grid_cells_for2(double L, double cut) {
  int n = (int)floor(L / cut);
  if (n < 1) n = 1;
  while (n > 1 && L / n < cut) --n;
  return n;
}

// scratch slots 24..43 belong to this file (observables.hip uses 0..13,
// ctx.hip 21..22, sweep.hip 23): descriptor grid 24..26, the insertion call's
// descriptor and overlap grids built together 27..29,
// rows / scores 30, targets / block partials 31, cumulative mass 32, gradient
// sums of the training workgroups 33, order of the training points 34,
// per-block insertion weights and hits 35, cumulative-mass block sums 36,
// grid-scan partials 37, voxel scores 38, score block reductions 39,
// free-voxel tile slots and list 40, tile counts, offsets and scan space 41,
// blocked-voxel flags 42, softmax statistics 43.
enum { L_GRID_A = 24, L_GRID_PAIR = 27, L_X = 30, L_T = 31, L_CDF = 32, L_GRAD = 33, L_ORDER = 34, L_PART = 35,
       L_BSUM = 36, L_SCANP = 37, L_F = 38, L_FRED = 39, L_LIST = 40, L_NFREE = 41, L_FLAG = 42,
       L_STATS = 43 };

void set_grid(NGrid &g, const RepHost &h, double cut, const int *start, const Pos *pos) {
  g.nx = grid_cells_for2(h.p.lx, cut);
  g.ny = grid_cells_for2(h.p.ly, cut);
  g.nz = grid_cells_for2(h.p.lz, cut);
  g.sx = h.p.lx / g.nx; g.sy = h.p.ly / g.ny; g.sz = h.p.lz / g.nz;
  g.ix = 1.0 / g.sx; g.iy = 1.0 / g.sy; g.iz = 1.0 / g.sz;
  g.lx = h.p.lx; g.ly = h.p.ly; g.lz = h.p.lz;
  g.start = start;
  g.p = pos;
}

// Descriptor grid (cut_a) and overlap grid (cut_b) of `replica` in one set
// of launches: the cache entry 1 of the context's grid cache, keyed by
// replica and configuration version (the cuts are the insertion call's
// constants).
int build_ngrid_pair(hsmc_gpu_ctx *ctx, int replica, double cut_a, double cut_b, NGrid &ga,
                     NGrid &gb) {
  const RepHost &h = ctx->reps[replica];
  const int N = h.p.n_part;
  const long Ca = (long)grid_cells_for2(h.p.lx, cut_a) * grid_cells_for2(h.p.ly, cut_a) *
                  grid_cells_for2(h.p.lz, cut_a);
  const long Cb = (long)grid_cells_for2(h.p.lx, cut_b) * grid_cells_for2(h.p.ly, cut_b) *
                  grid_cells_for2(h.p.lz, cut_b);
  const long C = Ca + Cb;
  if (C + 1 > (1L << 31) - 1 || 2L * N > (1L << 31) - 1) return HSMC_ERR_NOT_SUPPORTED;
  const bool cached = ctx->ngrid_replica[1] == replica && ctx->ngrid_version[1] == ctx->version &&
                      ctx->ngrid_cut[1] == cut_a + cut_b;
  const size_t cells = ((size_t)C + 4) & ~(size_t)3;  // keeps the int4 behind the counts aligned
  int *cnt = (int *)scratch(ctx, L_GRID_PAIR + 0, sizeof(int) * cells + sizeof(int4) * N);
  Pos *pos = (Pos *)scratch(ctx, L_GRID_PAIR + 1, sizeof(Pos) * 2 * (size_t)N);
  int *start = (int *)scratch(ctx, L_GRID_PAIR + 2, sizeof(int) * (C + 1));
  int *part = (int *)scratch(ctx, L_SCANP, sizeof(int) * scan_workspace_ints(C));
  if (!cnt || !pos || !start || !part) return HSMC_ERR_NO_MEMORY;
  int4 *at = (int4 *)(cnt + cells);  // each sphere's two cells and its rank in each
  set_grid(ga, h, cut_a, start, pos);
  set_grid(gb, h, cut_b, start + Ca, pos);
  if (cached) return HSMC_OK;
  const CellDims da{ga.nx, ga.ny, ga.nz, ga.ix, ga.iy, ga.iz};
  const CellDims db{gb.nx, gb.ny, gb.nz, gb.ix, gb.iy, gb.iz};
  const double *x = ctx->d_x + h.poff, *y = ctx->d_y + h.poff, *z = ctx->d_z + h.poff;
  HSMC_HIP(ctx, hipMemsetAsync(cnt, 0, sizeof(int) * (C + 1), ctx->stream));
  hipLaunchKernelGGL(k_grid_count_pair, dim3((N + 255) / 256), dim3(256), 0, ctx->stream, x, y, z,
                     N, da, db, (int)Ca, cnt, at);
  exclusive_scan(ctx->stream, cnt, (int)C, start, part, false);
  hipLaunchKernelGGL(k_grid_scatter_pair, dim3((N + 255) / 256), dim3(256), 0, ctx->stream, x, y,
                     z, N, at, start, pos);
  HSMC_HIP(ctx, hipGetLastError());
  ctx->ngrid_replica[1] = replica;
  ctx->ngrid_version[1] = ctx->version;
  ctx->ngrid_cut[1] = cut_a + cut_b;
  return HSMC_OK;
}

int build_ngrid(hsmc_gpu_ctx *ctx, int replica, double cut, int slot0, NGrid &g) {
  const RepHost &h = ctx->reps[replica];
  const int N = h.p.n_part;
  const int nx = grid_cells_for2(h.p.lx, cut), ny = grid_cells_for2(h.p.ly, cut),
            nz = grid_cells_for2(h.p.lz, cut);
  const long C = (long)nx * ny * nz;
  const int which = 0;  // entry 1 is the paired build's
  const bool cached = ctx->ngrid_replica[which] == replica &&
                      ctx->ngrid_version[which] == ctx->version && ctx->ngrid_cut[which] == cut;
  int *cnt = (int *)scratch(ctx, slot0 + 0, sizeof(int) * 2 * (C + 1) + sizeof(int) * N);
  Pos *pos = (Pos *)scratch(ctx, slot0 + 1, sizeof(Pos) * (size_t)N);
  int *start = (int *)scratch(ctx, slot0 + 2, sizeof(int) * (C + 1));
  int *part = (int *)scratch(ctx, L_SCANP, sizeof(int) * scan_workspace_ints(C));
  if (!cnt || !pos || !start || !part) return HSMC_ERR_NO_MEMORY;
  int *fill = cnt + (C + 1);
  int *cellof = fill + (C + 1);
  const double *x = ctx->d_x + h.poff, *y = ctx->d_y + h.poff, *z = ctx->d_z + h.poff;
  const double sx = h.p.lx / nx, sy = h.p.ly / ny, sz = h.p.lz / nz;
  g.nx = nx; g.ny = ny; g.nz = nz;
  g.sx = sx; g.sy = sy; g.sz = sz;
  g.ix = 1.0 / sx; g.iy = 1.0 / sy; g.iz = 1.0 / sz;
  g.lx = h.p.lx; g.ly = h.p.ly; g.lz = h.p.lz;
  g.start = start;
  g.p = pos;
  if (cached) return HSMC_OK;
  HSMC_HIP(ctx, hipMemsetAsync(cnt, 0, sizeof(int) * 2 * (C + 1), ctx->stream));
  hipLaunchKernelGGL(k_grid_count2, dim3((N + 255) / 256), dim3(256), 0, ctx->stream, x, y, z, N,
                     nx, ny, nz, g.ix, g.iy, g.iz, cnt, cellof);
  exclusive_scan(ctx->stream, cnt, (int)C, start, part, false);
  hipLaunchKernelGGL(k_grid_scatter2, dim3((N + 255) / 256), dim3(256), 0, ctx->stream, x, y, z,
                     N, cellof, start, fill, pos);
  HSMC_HIP(ctx, hipGetLastError());
  ctx->ngrid_replica[which] = replica;
  ctx->ngrid_version[which] = ctx->version;
  ctx->ngrid_cut[which] = cut;
  return HSMC_OK;
}

// The rows of n points.  From kSortRows points on, and at least one for each
// cell, in the order of their cells, kSortChunk points at a time (which bounds
// the workspace); their ranks lie where their targets will be.  A call with
// one pass over n points at N = 4000, unsorted and sorted (with the positions
// in three arrays; both 5 to 15 % faster as records): 2^15 points 104 and
// 118 us (the sort's three launches), 2^17 273 and 163, 2^20 1911 and 648; at
// N = 32000 128 and 121, 378 and 173, 2794 and 700; at N = 108, where the few
// cells' spheres stay in the first cache either way, 89 and 119, 154 and 162,
// 788 and 628.
constexpr long long kSortRows = 65536, kSortChunk = 1 << 20;

int launch_training_rows(hsmc_gpu_ctx *ctx, const NGrid &g, const Vox &vx, const TrainingPoints &point,
                         long long n, float far2, float beta, float *X, float *T) {
  const long C = (long)g.nx * g.ny * g.nz;
  if (n < kSortRows || C > n) {
    hipLaunchKernelGGL(k_training_rows, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, g, vx,
                       point, 0LL, n, (const int *)nullptr, far2, beta, X, T);
    HSMC_HIP(ctx, hipGetLastError());
    return HSMC_OK;
  }
  const size_t chunk = (size_t)std::min(n, kSortChunk);
  int *order = (int *)scratch(ctx, L_ORDER, sizeof(int) * (chunk + 2 * (size_t)C + 1 + (size_t)scan_workspace_ints(C)));
  if (!order) return HSMC_ERR_NO_MEMORY;
  int *cnt = order + chunk, *start = cnt + C, *part = start + C + 1;
  for (long long first = 0; first < n; first += kSortChunk) {
    const int m = (int)std::min(kSortChunk, n - first);
    int *rank = (int *)T + first;
    HSMC_HIP(ctx, hipMemsetAsync(cnt, 0, sizeof(int) * C, ctx->stream));
    hipLaunchKernelGGL(C <= kLdsCells ? k_training_count<true> : k_training_count<false>,
                       dim3((unsigned)((m + kSortThreads - 1) / kSortThreads)), dim3(kSortThreads), 0, ctx->stream,
                       g, vx, point, first, m, cnt, rank);
    exclusive_scan(ctx->stream, cnt, (int)C, start, part, false);
    const dim3 blocks((unsigned)((m + 255) / 256));
    hipLaunchKernelGGL(k_training_order, blocks, dim3(256), 0, ctx->stream, g, vx, point, first, m, start, rank,
                       order);
    hipLaunchKernelGGL(k_training_rows, blocks, dim3(256), 0, ctx->stream, g, vx, point, first, (long long)m,
                       order, far2, beta, X, T);
    HSMC_HIP(ctx, hipGetLastError());
  }
  return HSMC_OK;
}

// Workgroups of a training batch of n rows (64 rows each, the largest
// batches several times).
int grad_blocks(int n) { return (int)std::min(((long)n + 63) / 64, (long)kGradBlocks); }

constexpr double kDescCut = 1.5;  // descriptor grid side (sigma)

Vox make_vox(const RepHost &h, double voxel) {
  Vox v;
  v.mx = (int)ceil(h.p.lx / voxel);
  v.my = (int)ceil(h.p.ly / voxel);
  v.mz = (int)ceil(h.p.lz / voxel);
  v.vx = h.p.lx / v.mx;
  v.vy = h.p.ly / v.my;
  v.vz = h.p.lz / v.mz;
  v.V = (long)v.mx * v.my * v.mz;
  return v;
}

float far2_of(const NGrid &g) {
  const double s = std::min(g.sx, std::min(g.sy, g.sz));
  return (float)(s * s);
}

// Voxel scores into f, and per-block max / sum exp(f - max) into the scratch
// returned in *bred (*nblk blocks): the tiled kernel when every box edge
// exceeds 2 (tile extent + smin), else the per-voxel one.
int launch_scores(hsmc_gpu_ctx *ctx, const NGrid &g, const Vox &vx, const MlpDev *net, float *f,
                  float **bred, long *nblk) {
  const double smin = std::min(g.sx, std::min(g.sy, g.sz));
  const bool tiled = g.lx > 2.0 * ((TX - 1) * vx.vx + smin) * (1.0 + 1e-9) &&
                     g.ly > 2.0 * ((TY - 1) * vx.vy + smin) * (1.0 + 1e-9) &&
                     g.lz > 2.0 * ((TZ - 1) * vx.vz + smin) * (1.0 + 1e-9);
  const long nb = tiled ? (long)((vx.mx + TX - 1) / TX) * ((vx.my + TY - 1) / TY) * ((vx.mz + TZ - 1) / TZ)
                        : (vx.V + 255) / 256;
  float *b = (float *)scratch(ctx, L_FRED, sizeof(float) * 2 * (size_t)nb);
  if (!b) return HSMC_ERR_NO_MEMORY;
  if (tiled)
    hipLaunchKernelGGL(k_voxel_scores_tiled, dim3((unsigned)nb), dim3(256), 0, ctx->stream, g, vx,
                       far2_of(g), smin, net, f, b, b + nb);
  else
    hipLaunchKernelGGL(k_voxel_scores, dim3((unsigned)nb), dim3(256), 0, ctx->stream, g, vx,
                       far2_of(g), net, f, b, b + nb);
  HSMC_HIP(ctx, hipGetLastError());
  *bred = b;
  *nblk = nb;
  return HSMC_OK;
}

__global__ void k_iota(int *__restrict__ list, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) list[i] = (int)i;
}

// -inf for the voxels the flags mark as blocked (the proposal's scores as a
// caller sees them).
__global__ void k_mask_blocked(float *__restrict__ f, const unsigned char *__restrict__ flag,
                               long V) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < V && flag[i]) f[i] = -INFINITY;
}

// The proposal of one configuration: the byte flags of blocked voxels
// (k_mark_blocked), the list of free voxels (k_free_tiles, k_gather_free),
// the network's scores of the free voxels in f (k_voxel_scores_list), and the
// block partials of their softmax totals (with no free voxel the totals
// themselves: 0 and 1, so every voxel keeps the uniform part alone).  Where a voxel is too
// large for any exclusion, or too small for the marking kernel's 8
// candidates per axis, every voxel is free and scored.  Only the number of
// free voxels comes back to the host (it sizes the later launches).
struct Proposal {
  unsigned char *flag = nullptr;
  int *list = nullptr;
  const float *parts = nullptr;  // the scoring kernel's block partials
  long nparts = 0;
  long nfree = 0;
};

// `grid` builds the search grids and gives the descriptors' one; its launches
// run while the host waits for the number of free voxels.
template <class MakeGrid>
int launch_proposal_scores(hsmc_gpu_ctx *ctx, int replica, MakeGrid &&grid, const Vox &vx,
                           const MlpDev *net, float *f, Proposal *pr) {
  NGrid g;
  const double h = 0.5 * sqrt(vx.vx * vx.vx + vx.vy * vx.vy + vx.vz * vx.vz);
  const double r = 1.0 - h - 1e-9;
  // the marking kernel's 8 candidate voxels per axis must cover the centres
  // within r of a sphere (voxel_first), and each axis must have 8 voxels to
  // wrap over
  const double lim = 8.0 - 1e-6;
  const bool span_ok = 2.0 * r / vx.vx + 1.0 < lim && 2.0 * r / vx.vy + 1.0 < lim &&
                       2.0 * r / vx.vz + 1.0 < lim && vx.mx >= 8 && vx.my >= 8 && vx.mz >= 8;
  const long tiles = (long)((vx.mx + TX - 1) / TX) * ((vx.my + TY - 1) / TY) * ((vx.mz + TZ - 1) / TZ);
  // per tile: 256 free-voxel slots, then the packed list; the tile counts,
  // their prefix sum and the scan's workspace; a byte per voxel
  int *slots = (int *)scratch(ctx, L_LIST, sizeof(int) * ((size_t)tiles * 256 + (size_t)vx.V));
  int *cnt = (int *)scratch(ctx, L_NFREE,
                            sizeof(int) * (2 * (size_t)tiles + 1 + (size_t)scan_workspace_ints(tiles)));
  unsigned char *flag = (unsigned char *)scratch(ctx, L_FLAG, (size_t)vx.V);
  double *stats = (double *)scratch(ctx, L_STATS, sizeof(double) * 3);
  if (!slots || !cnt || !flag || !stats) return HSMC_ERR_NO_MEMORY;
  int *list = slots + (size_t)tiles * 256;
  pr->flag = flag;
  pr->list = list;
  HSMC_HIP(ctx, hipMemsetAsync(flag, 0, (size_t)vx.V, ctx->stream));
  if (!(r > 0.0) || !span_ok) {
    float *bred = nullptr;
    long nblk = 0;
    int st = grid(&g);
    if (st) return st;
    st = launch_scores(ctx, g, vx, net, f, &bred, &nblk);
    if (st) return st;
    hipLaunchKernelGGL(k_iota, dim3((unsigned)((vx.V + 255) / 256)), dim3(256), 0, ctx->stream, list,
                       vx.V);
    HSMC_HIP(ctx, hipGetLastError());
    pr->parts = bred;
    pr->nparts = nblk;
    pr->nfree = vx.V;
    return HSMC_OK;
  }
  const RepHost &rh = ctx->reps[replica];
  int *off = cnt + tiles;
  int *part = off + tiles + 1;
  const int N = rh.p.n_part;
  Box3 b3{rh.p.lx, rh.p.ly, rh.p.lz, 1.0 / vx.vx, 1.0 / vx.vy, 1.0 / vx.vz};
  hipLaunchKernelGGL(k_mark_blocked, dim3((unsigned)((N + 3) / 4)), dim3(256), 0, ctx->stream,
                     ctx->d_x + rh.poff, ctx->d_y + rh.poff, ctx->d_z + rh.poff, N, vx, b3, r, flag);
  hipLaunchKernelGGL(k_free_tiles, dim3((unsigned)((tiles + 3) / 4)), dim3(256), 0, ctx->stream, vx,
                     flag, slots, cnt, tiles);
  exclusive_scan(ctx->stream, cnt, (int)tiles, off, part, false);
  hipLaunchKernelGGL(k_gather_free, dim3((unsigned)((tiles + 3) / 4)), dim3(256), 0, ctx->stream,
                     slots, cnt, off, list, tiles, ctx->h_acc);
  HSMC_HIP(ctx, hipGetLastError());
  HSMC_HIP(ctx, hipEventRecord(ctx->ev0, ctx->stream));
  int st = grid(&g);
  if (st) return st;
  HSMC_HIP(ctx, hipEventSynchronize(ctx->ev0));
  const int nf = (int)ctx->h_acc[0];
  pr->nfree = nf;
  if (nf == 0) {
    hipLaunchKernelGGL(k_empty_stats, dim3(1), dim3(64), 0, ctx->stream, stats);
    HSMC_HIP(ctx, hipGetLastError());
    return HSMC_OK;
  }
  const long nb = ((long)nf + 255) / 256;
  float *b = (float *)scratch(ctx, L_FRED, sizeof(float) * 2 * (size_t)nb);
  if (!b) return HSMC_ERR_NO_MEMORY;
  // the softmax totals come from the scoring kernel's per-block max and sum of
  // exp(f - max) (each block's 256 list entries reduced in a fixed order),
  // combined in a fixed order: they depend only on the scores and the list
  hipLaunchKernelGGL(k_voxel_scores_list, dim3((unsigned)nb), dim3(256), 0, ctx->stream, g, vx,
                     far2_of(g), net, list, (int)nf, f, b, b + nb);
  HSMC_HIP(ctx, hipGetLastError());
  pr->parts = b;
  pr->nparts = nb;
  return HSMC_OK;
}

}  // namespace

extern "C" {

int hsmc_gpu_mlp_create(hsmc_gpu_ctx *ctx, hsmc_gpu_mlp **out, uint64_t seed) {
  if (!ctx || !out) return HSMC_ERR_BAD_ARG;
  hsmc_gpu_mlp *m = new hsmc_gpu_mlp();
  m->ctx = ctx;
  if (hipMalloc(&m->P, sizeof(float) * NPARAM) != hipSuccess ||
      hipMalloc(&m->G, sizeof(float) * NPARAM) != hipSuccess ||
      hipMalloc(&m->m1, sizeof(float) * NPARAM) != hipSuccess ||
      hipMalloc(&m->m2, sizeof(float) * NPARAM) != hipSuccess ||
      hipMalloc(&m->net, sizeof(MlpDev)) != hipSuccess ||
      hipMalloc(&m->loss, sizeof(float)) != hipSuccess) {
    hsmc_gpu_mlp_destroy(m);
    return HSMC_ERR_NO_MEMORY;
  }
  // He-uniform initial weights from Philox(seed), zero biases
  std::vector<float> p(NPARAM, 0.f);
  auto uni = [&](uint32_t i) {
    uint32_t u[4];
    philox4x32_10(i, 0x4D4C5000u, 0u, 0u, (uint32_t)seed, (uint32_t)(seed >> 32), u);
    return (float)(((double)u[0] + 0.5) * 0x1p-32 * 2.0 - 1.0);
  };
  const float a1 = sqrtf(6.f / NIN), a2 = sqrtf(6.f / NH);
  for (int i = 0; i < NIN * NH; ++i) p[OW1 + i] = a1 * uni(i);
  for (int i = 0; i < NH * NH; ++i) p[OW2 + i] = a2 * uni(10000 + i);
  for (int i = 0; i < NH; ++i) p[OW3 + i] = a2 * uni(20000 + i);
  int st = hsmc_gpu_mlp_set(m, p.data());
  if (st) {
    hsmc_gpu_mlp_destroy(m);
    return st;
  }
  *out = m;
  return HSMC_OK;
}

int hsmc_gpu_mlp_destroy(hsmc_gpu_mlp *m) {
  if (!m) return HSMC_OK;
  if (m->ctx) (void)hipStreamSynchronize(m->ctx->stream);
  void *b[] = {m->P, m->G, m->m1, m->m2, m->net, m->loss};
  for (void *x : b)
    if (x) (void)hipFree(x);
  delete m;
  return HSMC_OK;
}

int hsmc_gpu_mlp_forget(hsmc_gpu_mlp *m) {
  if (!m) return HSMC_ERR_BAD_ARG;
  m->sc_replica = -1;
  return HSMC_OK;
}

int hsmc_gpu_mlp_set(hsmc_gpu_mlp *m, const float *params) {
  if (!m || !params) return HSMC_ERR_BAD_ARG;
  hsmc_gpu_ctx *ctx = m->ctx;
  HSMC_HIP(ctx, hipMemcpyAsync(m->P, params, sizeof(float) * NPARAM, hipMemcpyHostToDevice, ctx->stream));
  HSMC_HIP(ctx, hipMemsetAsync(m->m1, 0, sizeof(float) * NPARAM, ctx->stream));
  HSMC_HIP(ctx, hipMemsetAsync(m->m2, 0, sizeof(float) * NPARAM, ctx->stream));
  HSMC_HIP(ctx, hipMemsetAsync(m->net, 0, sizeof(MlpDev), ctx->stream));
  hipLaunchKernelGGL(k_pack_net, dim3((NPARAM + 255) / 256), dim3(256), 0, ctx->stream, m->P, m->net);
  HSMC_HIP(ctx, hipGetLastError());
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  m->step = 0;
  m->sc_replica = -1;
  return HSMC_OK;
}

int hsmc_gpu_mlp_get(hsmc_gpu_mlp *m, float *params) {
  if (!m || !params) return HSMC_ERR_BAD_ARG;
  hsmc_gpu_ctx *ctx = m->ctx;
  HSMC_HIP(ctx, hipMemcpyAsync(params, m->P, sizeof(float) * NPARAM, hipMemcpyDeviceToHost, ctx->stream));
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return HSMC_OK;
}

int hsmc_gpu_mlp_forward(hsmc_gpu_mlp *m, const float *x, int n, float *y) {
  if (!m || n < 0 || (n > 0 && (!x || !y))) return HSMC_ERR_BAD_ARG;
  if (n == 0) return HSMC_OK;
  hsmc_gpu_ctx *ctx = m->ctx;
  float *dx = (float *)scratch(ctx, L_X, sizeof(float) * NIN * (size_t)n);
  float *dy = (float *)scratch(ctx, L_T, sizeof(float) * (size_t)n);
  if (!dx || !dy) return HSMC_ERR_NO_MEMORY;
  HSMC_HIP(ctx, hipMemcpyAsync(dx, x, sizeof(float) * NIN * (size_t)n, hipMemcpyHostToDevice, ctx->stream));
  hipLaunchKernelGGL(k_mlp_forward, dim3((unsigned)(((long)n + 255) / 256)), dim3(256), 0, ctx->stream, m->net, dx, n,
                     dy);
  HSMC_HIP(ctx, hipGetLastError());
  HSMC_HIP(ctx, hipMemcpyAsync(y, dy, sizeof(float) * (size_t)n, hipMemcpyDeviceToHost, ctx->stream));
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return HSMC_OK;
}

int hsmc_gpu_mlp_gradient(hsmc_gpu_mlp *m, const float *x, const float *t, int n, float *loss,
                          float *grad) {
  if (!m || n <= 0 || !x || !t) return HSMC_ERR_BAD_ARG;
  hsmc_gpu_ctx *ctx = m->ctx;
  float *dx = (float *)scratch(ctx, L_X, sizeof(float) * NIN * (size_t)n);
  float *dt = (float *)scratch(ctx, L_T, sizeof(float) * (size_t)n);
  if (!dx || !dt) return HSMC_ERR_NO_MEMORY;
  HSMC_HIP(ctx, hipMemcpyAsync(dx, x, sizeof(float) * NIN * (size_t)n, hipMemcpyHostToDevice, ctx->stream));
  HSMC_HIP(ctx, hipMemcpyAsync(dt, t, sizeof(float) * (size_t)n, hipMemcpyHostToDevice, ctx->stream));
  float *part = (float *)scratch(ctx, L_GRAD, sizeof(float) * kGradStride * grad_blocks(n));
  if (!part) return HSMC_ERR_NO_MEMORY;
  HSMC_HIP(ctx, hipMemsetAsync(m->loss, 0, sizeof(float), ctx->stream));
  hipLaunchKernelGGL(k_mlp_train_step, dim3(grad_blocks(n)), dim3(256), 0, ctx->stream, m->net, dx,
                     dt, n, 1.0f / n, part);
  hipLaunchKernelGGL(k_reduce_grad<false>, dim3(NPARAM / 64 + 1), dim3(256), 0, ctx->stream, part,
                     grad_blocks(n), m->P, m->G, m->m1, m->m2, 0.f, 0.f, 0.f, 0.f, 1.f, 1.f, m->net,
                     m->loss);
  HSMC_HIP(ctx, hipGetLastError());
  float l = 0.f;
  HSMC_HIP(ctx, hipMemcpyAsync(&l, m->loss, sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
  if (grad)
    HSMC_HIP(ctx, hipMemcpyAsync(grad, m->G, sizeof(float) * NPARAM, hipMemcpyDeviceToHost, ctx->stream));
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (loss) *loss = l / n;
  return HSMC_OK;
}

int hsmc_gpu_point_descriptors(hsmc_gpu_ctx *ctx, int replica, const double *xyz, int m,
                               float *desc) {
  if (!ctx || replica < 0 || replica >= ctx->R || m < 0 || (m > 0 && (!xyz || !desc)))
    return HSMC_ERR_BAD_ARG;
  if (m == 0) return HSMC_OK;
  NGrid g;
  int st = build_ngrid(ctx, replica, kDescCut, L_GRID_A, g);
  if (st) return st;
  double *dq = (double *)scratch(ctx, L_X, sizeof(double) * 3 * (size_t)m);
  float *dd = (float *)scratch(ctx, L_T, sizeof(float) * NIN * (size_t)m);
  if (!dq || !dd) return HSMC_ERR_NO_MEMORY;
  HSMC_HIP(ctx, hipMemcpyAsync(dq, xyz, sizeof(double) * 3 * m, hipMemcpyHostToDevice, ctx->stream));
  hipLaunchKernelGGL(k_point_descriptors, dim3((m + 255) / 256), dim3(256), 0, ctx->stream, g, dq,
                     m, far2_of(g), dd);
  HSMC_HIP(ctx, hipGetLastError());
  HSMC_HIP(ctx, hipMemcpyAsync(desc, dd, sizeof(float) * NIN * m, hipMemcpyDeviceToHost, ctx->stream));
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return HSMC_OK;
}

int hsmc_gpu_mlp_train(hsmc_gpu_mlp *m, int replica, double voxel, uint64_t seed, uint64_t sample,
                       int64_t n_points, int epochs, int batch, float lr, float beta,
                       float *final_loss) {
  if (!m || n_points <= 0 || epochs <= 0 || batch < 64 || !(voxel > 0.0)) return HSMC_ERR_BAD_ARG;
  hsmc_gpu_ctx *ctx = m->ctx;
  if (replica < 0 || replica >= ctx->R) return HSMC_ERR_BAD_ARG;
  NGrid g;
  int st = build_ngrid(ctx, replica, kDescCut, L_GRID_A, g);
  if (st) return st;
  const Vox vx = make_vox(ctx->reps[replica], voxel);
  float *X = (float *)scratch(ctx, L_X, sizeof(float) * NIN * (size_t)n_points);
  float *T = (float *)scratch(ctx, L_T, sizeof(float) * (size_t)n_points);
  if (!X || !T) return HSMC_ERR_NO_MEMORY;
  st = launch_training_rows(ctx, g, vx, TrainingPoints{(uint32_t)seed, (uint32_t)(seed >> 32), sample},
                            n_points, far2_of(g), beta, X, T);
  if (st) return st;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const int gb = grad_blocks((int)std::min<int64_t>(batch, n_points));
  float *part = (float *)scratch(ctx, L_GRAD, sizeof(float) * kGradStride * gb);
  if (!part) return HSMC_ERR_NO_MEMORY;
  for (int e = 0; e < epochs; ++e) {
    HSMC_HIP(ctx, hipMemsetAsync(m->loss, 0, sizeof(float), ctx->stream));
    for (int64_t b0 = 0; b0 < n_points; b0 += batch) {
      const int nb = (int)std::min<int64_t>(batch, n_points - b0);
      hipLaunchKernelGGL(k_mlp_train_step, dim3(grad_blocks(nb)), dim3(256), 0, ctx->stream, m->net,
                         X + (size_t)b0 * NIN, T + b0, nb, 1.0f / nb, part);
      ++m->step;
      const float c1 = 1.f - powf(b1, (float)m->step), c2 = 1.f - powf(b2, (float)m->step);
      hipLaunchKernelGGL(k_reduce_grad<true>, dim3(NPARAM / 64 + 1), dim3(256), 0, ctx->stream, part,
                         grad_blocks(nb), m->P, m->G, m->m1, m->m2, lr, b1, b2, eps, c1, c2, m->net,
                         m->loss);
    }
    HSMC_HIP(ctx, hipGetLastError());
  }
  float last = 0.f;  // the last epoch's sum
  HSMC_HIP(ctx, hipMemcpyAsync(&last, m->loss, sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (final_loss) *final_loss = last / (float)n_points;
  return HSMC_OK;
}

int hsmc_gpu_widom_learned(hsmc_gpu_mlp *m, int replica, double voxel, double mix, uint64_t seed,
                           uint64_t sample, int64_t n, double *estimate, int64_t *n_done,
                           int64_t *hits) {
  if (!m || !estimate || n <= 0 || n > (1LL << 30) || !(mix >= 0.0 && mix < 1.0) || !(voxel > 0.0))
    return HSMC_ERR_BAD_ARG;
  hsmc_gpu_ctx *ctx = m->ctx;
  if (replica < 0 || replica >= ctx->R) return HSMC_ERR_BAD_ARG;
  const Vox vx = make_vox(ctx->reps[replica], voxel);
  if (vx.V > (1L << 31) - 1) return HSMC_ERR_NOT_SUPPORTED;
  NGrid g1;
  auto grids = [&](NGrid *g) { return build_ngrid_pair(ctx, replica, kDescCut, 1.0 + 1e-9, *g, g1); };
  float *f = (float *)scratch(ctx, L_F, sizeof(float) * (size_t)vx.V);
  const long nblk_ins = (long)((n + 255) / 256);
  double *part = (double *)scratch(ctx, L_PART, (sizeof(double) + sizeof(unsigned int)) * (size_t)nblk_ins);
  if (!f || !part) return HSMC_ERR_NO_MEMORY;
  unsigned int *hpart = (unsigned int *)(part + nblk_ins);
  const bool scores_ok = m->sc_replica == replica && m->sc_version == ctx->version &&
                         m->sc_step == m->step && m->sc_voxel == voxel &&
                         m->sc_stamp == ctx->score_stamp;
  Proposal pr;
  int st = HSMC_OK;
  if (scores_ok) {
    NGrid g;
    st = grids(&g);
    if (st) return st;
  } else {
    // the shared buffers are overwritten: no network's cache stays valid, and
    // this one's holds again once its last kernel is launched
    m->sc_replica = -1;
    ++ctx->score_stamp;
    st = launch_proposal_scores(ctx, replica, grids, vx, m->net, f, &pr);
    if (st) return st;
  }
  // the cached proposal's flags and free list (the same scratch the scoring
  // wrote; the stamp check above guarantees nobody rewrote it since)
  const long tiles = (long)((vx.mx + TX - 1) / TX) * ((vx.my + TY - 1) / TY) * ((vx.mz + TZ - 1) / TZ);
  int *slots = (int *)scratch(ctx, L_LIST, sizeof(int) * ((size_t)tiles * 256 + (size_t)vx.V));
  unsigned char *flag = (unsigned char *)scratch(ctx, L_FLAG, (size_t)vx.V);
  double *stats = (double *)scratch(ctx, L_STATS, sizeof(double) * 3);
  if (!slots || !flag || !stats) return HSMC_ERR_NO_MEMORY;
  const int *list = slots + (size_t)tiles * 256;
  const long nfree = scores_ok ? m->sc_nfree : pr.nfree;
  const long ncdf = std::max(1L, (nfree + 4095) / 4096);
  double *cdf = (double *)scratch(ctx, L_CDF, sizeof(double) * (size_t)std::max(1L, nfree));
  double *bsum = (double *)scratch(ctx, L_BSUM, sizeof(double) * (size_t)(ncdf + 1));
  if (!cdf || !bsum) return HSMC_ERR_NO_MEMORY;
  const bool new_mass = !scores_ok || m->sc_mix != mix;
  if (new_mass) m->sc_replica = -1;
  if (new_mass && nfree > 0) {
    const float *parts = pr.parts;
    if (parts && pr.nparts > kStatsParts) {
      hipLaunchKernelGGL(k_softmax_stats, dim3(1), dim3(256), 0, ctx->stream, parts, pr.nparts, stats);
      parts = nullptr;
    }
    hipLaunchKernelGGL(k_cdf_local, dim3((unsigned)ncdf), dim3(1024), 0, ctx->stream, f, list, nfree,
                       parts, pr.nparts, stats, mix, cdf, bsum);
    const dim3 add_blocks((unsigned)((nfree + 255) / 256));
    if (ncdf <= kScanWave) {
      hipLaunchKernelGGL(k_cdf_add<true>, add_blocks, dim3(256), 0, ctx->stream, cdf, nfree, bsum, (int)ncdf,
                         bsum + ncdf);
    } else {
      hipLaunchKernelGGL(k_cdf_blocks, dim3(1), dim3(1024), 0, ctx->stream, bsum, (int)ncdf);
      hipLaunchKernelGGL(k_cdf_add<false>, add_blocks, dim3(256), 0, ctx->stream, cdf, nfree, bsum, (int)ncdf,
                         bsum + ncdf);
    }
    HSMC_HIP(ctx, hipGetLastError());
  }
  m->sc_replica = replica;
  m->sc_version = ctx->version;
  m->sc_step = m->step;
  m->sc_voxel = voxel;
  m->sc_nfree = nfree;
  m->sc_mix = mix;
  if (new_mass) m->sc_stamp = ++ctx->score_stamp;
  // the network mass's total: the scan's last entry, or 0 with no free voxel
  const double *total = nfree > 0 ? bsum + ncdf : stats + 2;
  // one uniform offset per call for the systematic sample
  uint32_t u[4];
  philox4x32_10(0u, 0u, (uint32_t)sample, 0x4C530000u | (uint32_t)((sample >> 32) & 0xFFFFu),
                (uint32_t)seed, (uint32_t)(seed >> 32), u);
  const double u0 = (double)u[0] * 0x1p-32;
  hipLaunchKernelGGL(k_insert, dim3((unsigned)nblk_ins), dim3(256), 0, ctx->stream, g1, vx,
                     cdf, list, nfree, total, (long)n, u0, f, flag, stats, mix,
                     (uint32_t)seed, (uint32_t)(seed >> 32), (unsigned long long)sample, part, hpart);
  hipLaunchKernelGGL(k_sum_fixed, dim3(1), dim3(256), 0, ctx->stream, part, hpart, nblk_ins, ctx->h_acc);
  HSMC_HIP(ctx, hipGetLastError());
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  *estimate = __builtin_bit_cast(double, ctx->h_acc[0]);
  if (n_done) *n_done = n;
  if (hits) *hits = (int64_t)ctx->h_acc[1];
  return HSMC_OK;
}

int hsmc_gpu_voxel_scores(hsmc_gpu_mlp *m, int replica, double voxel, float *scores, int64_t cap,
                          int64_t *n_voxels) {
  if (!m || !(voxel > 0.0) || !n_voxels) return HSMC_ERR_BAD_ARG;
  hsmc_gpu_ctx *ctx = m->ctx;
  if (replica < 0 || replica >= ctx->R) return HSMC_ERR_BAD_ARG;
  const Vox vx = make_vox(ctx->reps[replica], voxel);
  *n_voxels = vx.V;
  if (!scores) return HSMC_OK;
  if (cap < vx.V) return HSMC_ERR_BAD_ARG;
  NGrid g;
  int st = build_ngrid(ctx, replica, kDescCut, L_GRID_A, g);
  if (st) return st;
  float *f = (float *)scratch(ctx, L_F, sizeof(float) * (size_t)vx.V);
  if (!f) return HSMC_ERR_NO_MEMORY;
  // the shared score buffer is overwritten: no network's cache stays valid
  ++ctx->score_stamp;
  m->sc_replica = -1;
  float *bred = nullptr;
  long nblk = 0;
  st = launch_scores(ctx, g, vx, m->net, f, &bred, &nblk);
  if (st) return st;
  HSMC_HIP(ctx, hipMemcpyAsync(scores, f, sizeof(float) * vx.V, hipMemcpyDeviceToHost, ctx->stream));
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return HSMC_OK;
}

int hsmc_gpu_proposal_scores(hsmc_gpu_mlp *m, int replica, double voxel, float *scores,
                             int64_t cap, int64_t *n_voxels, int64_t *n_free) {
  if (!m || !(voxel > 0.0) || !n_voxels) return HSMC_ERR_BAD_ARG;
  hsmc_gpu_ctx *ctx = m->ctx;
  if (replica < 0 || replica >= ctx->R) return HSMC_ERR_BAD_ARG;
  const Vox vx = make_vox(ctx->reps[replica], voxel);
  *n_voxels = vx.V;
  if (!scores) return HSMC_OK;
  if (cap < vx.V) return HSMC_ERR_BAD_ARG;
  if (vx.V > (1L << 31) - 1) return HSMC_ERR_NOT_SUPPORTED;
  float *f = (float *)scratch(ctx, L_F, sizeof(float) * (size_t)vx.V);
  if (!f) return HSMC_ERR_NO_MEMORY;
  // the shared score buffer is overwritten: no network's cache stays valid
  ++ctx->score_stamp;
  m->sc_replica = -1;
  Proposal pr;
  int st = launch_proposal_scores(
      ctx, replica, [&](NGrid *g) { return build_ngrid(ctx, replica, kDescCut, L_GRID_A, *g); }, vx, m->net, f, &pr);
  if (st) return st;
  hipLaunchKernelGGL(k_mask_blocked, dim3((unsigned)((vx.V + 255) / 256)), dim3(256), 0,
                     ctx->stream, f, pr.flag, vx.V);
  HSMC_HIP(ctx, hipGetLastError());
  if (n_free) *n_free = pr.nfree;
  HSMC_HIP(ctx, hipMemcpyAsync(scores, f, sizeof(float) * vx.V, hipMemcpyDeviceToHost, ctx->stream));
  HSMC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return HSMC_OK;
}

}  // extern "C"
