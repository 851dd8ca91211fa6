// heat_kernels.h -- kernels and launch sequence of the differentiable temperature field,
// shared by every entry point of it (each brings its own device buffers).
#pragma once
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdio.h>

#include <algorithm>
#include <vector>

#include "../../include/amcafe.h"
#include "gl25.h"

namespace amcafe_heat {

static __constant__ double kHx[AMC_GL25_N] = AMC_GL25_X;
static __constant__ double kHw[AMC_GL25_N] = AMC_GL25_W;

struct Src {  // one parameter set
  double P, v, eta, sigma;
};
struct Geo {
  int nx, ny, nz;
  double dx, xs, ys, zs, dt, T0, tL, width, k, alpha, h;
};

// The rise of voxel (x, y, z) at time t is sum_q A_q(y, z) G_q(x, t) over the 25 quadrature nodes,
//   A_q = amp_q exp(-dy^2/D1_q - dz^2/(4 alpha tau_q)),  G_q = exp(-(x - x_laser(t) + v tau_q)^2/D1_q),
// a matrix product over q of all (y, z) rows with all (x, t) columns of a segment; so are the sums
// for its derivatives in v and sigma, with
//   G_q dx_q (t - tau_q) 2/D1_q,   A_q (k1_q + k2_q dy^2) with G_q, and G_q k2_q dx_q^2 with A_q.
// A wave takes 32 rows (its A in registers) and columns 32 at a time: the columns' G go to LDS (one
// exponential per node and column, shared by the block's four waves), the products run on the
// matrix cores (32x32x2 FP32, 13 steps of two nodes), and each lane evaluates the indicators of its
// 16 results.  Most of a domain is too cold to count at most times (8% of the 32x32 tiles of
// 256x256x64 voxels and 2000 steps are not), so a block first bounds its tiles, one per lane, and
// goes through those that can count; the rows of a wave are a compact patch of 8 x 4 (y, z), which
// leaves fewer of them than 32 in a line.  Evaluating the nodes' exponentials for every voxel-step
// took 50 exponentials each: that domain's loss 45.0 -> 2.7 ms, loss and gradient 60.0 -> 4.1 ms.  The
// matrix products (26 of 64 cycles per 1024 results) and the indicators (about as much) bound it.
constexpr int NQ = AMC_GL25_N, KP = 26;  // nodes, padded to pairs (the padding's A is 0)
constexpr int RT = 32, CT = 32;          // rows and columns of a wave's tile
constexpr int HB = 256, ROWS = RT * (HB / 64);

// Per-set constants of the nodes, in LDS (FP64: the positions' differences are taken before
// rounding to FP32).
struct NodeK {
  double vtau[KP], tau[KP];
  float iD1[KP], iDz[KP], k1[KP], k2[KP], amp[KP];
};
__device__ inline void node_consts(const Geo& g, const Src& s, NodeK* K, int i) {
  const double C = s.eta * s.P / (M_PI * (g.k / g.alpha) * sqrt(4 * M_PI * g.alpha));
  const double s2 = s.sigma * s.sigma;
  const double tau = g.h * (1 - kHx[i]), W = g.h * kHw[i];
  const double A = 2 * g.alpha * tau + s2, D1 = 2 * A;
  K->tau[i] = tau;
  K->vtau[i] = s.v * tau;
  K->iD1[i] = (float)(1 / D1);
  K->iDz[i] = (float)(1 / (4 * g.alpha * tau));
  K->k1[i] = (float)(-2 * s.sigma / A);
  K->k2[i] = (float)(4 * s.sigma / (D1 * D1));
  K->amp[i] = (float)(W * C / (sqrt(tau) * A));
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr float kLog2e = 1.44269504088896340736f;
__device__ inline float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }
// exp(x) for x <= 0: 2^(x log2 e) with the product's rounding error carried
__device__ inline float exp_neg(float x) {
  x = x < -200.0f ? -200.0f : x;  // (0 either way; keeps -inf out of the error term)
  const float h = x * kLog2e;
  const float l = fmaf(x, kLog2e, -h) + x * 1.925963033500011e-8f;
  return exp2_hw(h) * fmaf(l, 0.693147180559945f, 1.0f);
}
// 1 / (1 + exp(-d/width)) with d = T - tL (not NaN); ic = -log2(e)/width
__device__ inline float indicator(float d, float ic) {
  const float x = 1.0f + exp2_hw(fminf(d * ic, 126.0f));
  const float y = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, y, 1.0f), y, y);
}

// Fixed-order block sum in FP64 (butterfly within each wave, then the waves in order; a wave is a row of
// the block).
__device__ inline double block_sum(double v, double* sh) {
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();
  if (threadIdx.x == 0) sh[threadIdx.y] = v;
  __syncthreads();
  double t = 0;
  for (int q = 0; q < HB / 64; ++q) t += sh[q];
  return t;
}

// Row r of row tile `tile`: a patch of 8 x 4 (y, z), or 32 in a line (Shape::patch, see there).
// Returns false outside the domain.
__device__ inline bool row_of(const Geo& g, int patch, int tile, int r, int* y, int* z) {
  if (patch) {
    const int ty = (g.ny + 7) >> 3, tz = tile / ty;
    *y = 8 * (tile - tz * ty) + (r & 7);
    *z = 4 * tz + (r >> 3);
    return *y < g.ny && *z < g.nz;
  }
  const int row = tile * RT + r;
  *z = row / g.ny;
  *y = row - *z * g.ny;
  return row < g.ny * g.nz;
}
// Step and position of column `col` of a segment.
__device__ inline void col_of(const Geo& g, long long ncol, long long col, int* m, int* i) {
  if (ncol < (1ll << 31)) {  // (a 64-bit division takes as long as four nodes of a column)
    *m = (unsigned)col / (unsigned)g.nx;
    *i = (unsigned)col - (unsigned)*m * (unsigned)g.nx;
  } else {
    *m = (int)(col / g.nx);
    *i = (int)(col - (long long)*m * g.nx);
  }
}

// Grid: x = group of four row tiles (turned by y), y = share of the columns (column tiles y, y + gridDim.y, ...: the
// hot ones move with the source, so every share has its part of them), z = instance.  `part` holds 5
// sums (loss, gradient) per block, overwritten by the first segment, accumulated by later ones in
// launch order, so the result does not depend on scheduling.
//
// Skipped, as their terms are below 2e-35 (indicator values below e^-40): tiles whose rises all stay
// below the cut tL - 40 width - T0 for both sets, by the bound sum_q max A_q max G_q (A at the rows'
// least offsets, G at the columns' least distance from each node) or by the rises themselves.
template <bool GRAD>
__global__ __launch_bounds__(HB, GRAD ? 3 : 4) void k_heat(Geo g, const Src* S, const Src* Tg, int step0, int nsteps,
                                                        int ctiles, int patch, float* part, int first, unsigned long long* evals) {
  constexpr int NM = GRAD ? 4 : 2;  // column matrices: G of theta and of the target, and the derivatives'
  __shared__ NodeK Ks, Kt;
  __shared__ float sG[2][NM][KP * CT];
  __shared__ float sAm[HB / 64][2][32];  // per wave, set and node: bound on A over the wave's rows
  __shared__ unsigned long long smask[HB / 64];
  __shared__ double sh[HB / 64];
  __shared__ int sodd;
  const Src s = S[blockIdx.z], tgt = Tg[blockIdx.z];
  const int lane = threadIdx.x, w = threadIdx.y, tid = 64 * w + lane;
  const long long ncol = (long long)nsteps * g.nx;
  const int ntile = (int)((ncol + CT - 1) / CT);
  // Consecutive workgroups go to the chip's eight dies in turn, and the hot groups of a domain lie a
  // multiple of eight apart: each share starts with another group, or two dies would do all the work.
  const int group = (int)((blockIdx.x + blockIdx.y) % gridDim.x);
  float* slot = part + 5 * ((size_t)(blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + group);
  if (tid == 0) sodd = 0;
  __syncthreads();
  const float off = (float)(g.T0 - g.tL), ic = -kLog2e / (float)g.width;
  if (w < 2 && lane < KP) {  // wave 0: theta's nodes, wave 1: the target's
    NodeK& K = w ? Kt : Ks;
    if (lane < NQ) {
      node_consts(g, w ? tgt : s, &K, lane);
      // parameters that are not finite: no tile is skipped, and NaN goes through
      if (!(fabs(K.vtau[lane]) + fabs(K.tau[lane]) + fabs((double)K.iD1[lane]) + fabs((double)K.iDz[lane]) +
                fabs((double)K.amp[lane]) + fabs((double)off) + fabs((double)ic) + fabs(g.xs) + fabs(g.ys) + fabs(g.zs) +
                fabs(g.dt) + fabs(g.dx) <
            1e30))
        sodd = 1;
    } else {
      K.amp[lane] = K.iD1[lane] = K.iDz[lane] = K.k1[lane] = K.k2[lane] = 0.0f;
      K.vtau[lane] = K.tau[lane] = 0.0;
    }
  }
  __syncthreads();
  const bool odd = sodd != 0;
  const float cut = (float)(g.tL - 40 * g.width - g.T0), cutm = cut - 1e-3f * fabsf(cut);
  // the wave's rows: lane i and lane i + 32 hold row i's even and odd nodes
  float as[KP / 2], at[KP / 2], a2[GRAD ? KP / 2 : 1];
  int y, z;
  const bool in_row = row_of(g, patch, group * (HB / 64) + w, lane & 31, &y, &z);
  const int nrow = __popcll(__ballot(in_row) & 0xffffffffull);
  const double dyd = (y + 0.5) * g.dx - g.ys, dzd = (z + 0.5) * g.dx - g.zs;
  const float dy2 = (float)(dyd * dyd), dz2 = (float)(dzd * dzd);
  bool alive;  // some column could count for the wave's rows
  {
    float my = in_row ? dy2 : __builtin_inff(), mz = in_row ? dz2 : __builtin_inff();
    for (int o = 16; o >= 1; o >>= 1) {
      my = fminf(my, __shfl_xor(my, o));
      mz = fminf(mz, __shfl_xor(mz, o));
    }
    const NodeK& K = lane < 32 ? Ks : Kt;
    const int q = lane & 31;
    float am = q < NQ && nrow ? fabsf(K.amp[q]) * exp_neg(-my * K.iD1[q] - mz * K.iDz[q]) : 0.0f;
    sAm[w][lane >> 5][q] = am;
    for (int o = 16; o >= 1; o >>= 1) am += __shfl_xor(am, o);
    alive = nrow && (odd || __any(!(am < cutm)));
  }
  if (!__syncthreads_or(alive)) {
    if (tid < 5 && first) slot[tid] = 0.0f;
    return;
  }
  bool rows = false;  // as, at and a2 are there
  // a column's G, for both sets: thread = column tid & 31, nodes tid >> 5, + 8, ...
  auto columns = [&](int tile, int buf) {
    const int c = tid & 31;
    const long long col = (long long)tile * CT + c;
    const bool in = col < ncol;
    int m, i;
    col_of(g, ncol, in ? col : 0, &m, &i);
    const double t = (step0 + 1 + m) * g.dt, x0 = (i + 0.5) * g.dx - g.xs;
    const double cs = x0 - s.v * t, ct = x0 - tgt.v * t;  // x - x_laser(t)
    for (int q = tid >> 5; q < KP; q += HB / 32) {
      const float ds = (float)(cs + Ks.vtau[q]), dt = (float)(ct + Kt.vtau[q]);
      const float gs = in ? exp_neg(-ds * ds * Ks.iD1[q]) : 0.0f;
      sG[buf][0][q * CT + c] = gs;
      sG[buf][1][q * CT + c] = in ? exp_neg(-dt * dt * Kt.iD1[q]) : 0.0f;
      if constexpr (GRAD) {
        sG[buf][2][q * CT + c] = gs * (ds * (float)(t - Ks.tau[q]) * (2.0f * Ks.iD1[q]));
        sG[buf][3][q * CT + c] = gs * (Ks.k2[q] * (ds * ds));
      }
    }
  };
  double loss = 0, g0 = 0, g1 = 0, g3 = 0;
  unsigned long long ne = 0;
  for (int base = 0; base < ctiles; base += 8) {
    // ---- can tile base + lane/8 of the share count for the wave's rows? (nodes lane%8, + 8, ...)
    const int sub = lane & 7;
    const long long tl = blockIdx.y + (long long)(base + (lane >> 3)) * gridDim.y;
    const bool there = base + (lane >> 3) < ctiles && tl < ntile;
    float sum[2] = {0.0f, 0.0f};
    if (alive && there) {
      int m0, m1, i0, i1;
      col_of(g, ncol, tl * CT, &m0, &i0);
      col_of(g, ncol, min(tl * CT + CT, ncol) - 1, &m1, &i1);
      if (m0 != m1) {
        i0 = 0;
        i1 = g.nx - 1;
      }
      const double xa = (i0 + 0.5) * g.dx - g.xs, xb = (i1 + 0.5) * g.dx - g.xs;
      const double ta = (step0 + 1 + m0) * g.dt, tb = (step0 + 1 + m1) * g.dt;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const NodeK& K = u ? Kt : Ks;
        const double v = u ? tgt.v : s.v;
        const double lo = xa - fmax(v * ta, v * tb), hi = xb - fmin(v * ta, v * tb);
        for (int q = sub; q < KP; q += 8) {
          const float d = fmaxf(0.0f, fmaxf((float)(lo + K.vtau[q]), (float)-(hi + K.vtau[q])));
          sum[u] += sAm[w][u][q] * exp2_hw(-kLog2e * (d * d * K.iD1[q]));
        }
      }
    }
    for (int o = 4; o >= 1; o >>= 1) {
      sum[0] += __shfl_xor(sum[0], o);
      sum[1] += __shfl_xor(sum[1], o);
    }
    const bool need = alive && there && (odd || !(sum[0] < cutm && sum[1] < cutm));
    const unsigned long long mask = __ballot(need && sub == 0);  // bit 8 i: tile base + i
    if (lane == 0) smask[w] = mask;
    __syncthreads();
    unsigned long long rest = 0;
    for (int q = 0; q < HB / 64; ++q) rest |= smask[q];
    const unsigned rlo = __builtin_amdgcn_readfirstlane((unsigned)rest);
    const unsigned rhi = __builtin_amdgcn_readfirstlane((unsigned)(rest >> 32));
    rest = ((unsigned long long)rhi << 32) | rlo;
    if (rest != 0 && !rows) {
      rows = true;
#pragma unroll
      for (int p = 0; p < KP / 2; ++p) {
        const int q = 2 * p + (lane >> 5);
        as[p] = in_row ? Ks.amp[q] * exp_neg(-dy2 * Ks.iD1[q] - dz2 * Ks.iDz[q]) : 0.0f;
        at[p] = in_row ? Kt.amp[q] * exp_neg(-dy2 * Kt.iD1[q] - dz2 * Kt.iDz[q]) : 0.0f;
        if (GRAD) a2[p] = as[p] * (Ks.k1[q] + Ks.k2[q] * dy2);
      }
    }
    // ---- the tiles that can, for any of the waves
    int next = rest ? __builtin_ctzll(rest) : -1, buf = 0;
    if (next >= 0) columns(blockIdx.y + (base + (next >> 3)) * (int)gridDim.y, 0);
    while (next >= 0) {
      const int cur = next;
      rest &= rest - 1;
      next = rest ? __builtin_ctzll(rest) : -1;
      __syncthreads();  // this tile's columns are there; the other buffer's readers are done
      if (next >= 0) columns(blockIdx.y + (base + (next >> 3)) * (int)gridDim.y, buf ^ 1);
      if ((mask >> cur) & 1ull) {
        f32x16 xs = {}, xt = {}, xv = {}, xg = {};
#pragma unroll
        for (int p = 0; p < KP / 2; ++p) {
          xs = __builtin_amdgcn_mfma_f32_32x32x2f32(as[p], sG[buf][0][p * 64 + lane], xs, 0, 0, 0);
          xt = __builtin_amdgcn_mfma_f32_32x32x2f32(at[p], sG[buf][1][p * 64 + lane], xt, 0, 0, 0);
        }
        float mx = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, fmaxf(xs[r], xt[r]));
        if (__any(mx >= cut) || odd) {
          if constexpr (GRAD) {
#pragma unroll
            for (int p = 0; p < KP / 2; ++p) {
              xv = __builtin_amdgcn_mfma_f32_32x32x2f32(as[p], sG[buf][2][p * 64 + lane], xv, 0, 0, 0);
              xg = __builtin_amdgcn_mfma_f32_32x32x2f32(a2[p], sG[buf][0][p * 64 + lane], xg, 0, 0, 0);
              xg = __builtin_amdgcn_mfma_f32_32x32x2f32(as[p], sG[buf][3][p * 64 + lane], xg, 0, 0, 0);
            }
          }
          const long long c0 = (blockIdx.y + (long long)(base + (cur >> 3)) * gridDim.y) * CT;
          ne += (unsigned)nrow * (unsigned long long)min((long long)CT, ncol - c0);
          float l = 0, l0 = 0, l1 = 0, l3 = 0;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float a = indicator(xs[r] + off, ic), b = indicator(xt[r] + off, ic);
            const float df = a - b;
            l = fmaf(df, df, l);
            if constexpr (GRAD) {
              const float lam = df * (a * (1.0f - a));  // dloss/dT: times 2/width at the end
              l0 = fmaf(lam, xs[r], l0);
              l1 = fmaf(lam, xv[r], l1);
              l3 = fmaf(lam, xg[r], l3);
            }
          }
          if (odd) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
              if (xs[r] != xs[r] || xt[r] != xt[r] || off != off || ic != ic) l = l0 = l1 = l3 = __builtin_nanf("");
          }
          loss += l;
          if constexpr (GRAD) {
            g0 += l0;
            g1 += l1;
            g3 += l3;
          }
        }
      }
      buf ^= 1;
    }
    __syncthreads();
  }
  if (evals && ne && lane == 0) atomicAdd(evals, ne);
  if (!__syncthreads_or(ne != 0)) {
    if (tid < 5 && first) slot[tid] = 0.0f;
    return;
  }
  const double sc = 2 / g.width;
  const double t0 = block_sum(loss, sh);
  double t1 = 0, t2 = 0, t3 = 0;
  if (GRAD) {
    t1 = block_sum(g0, sh);
    t2 = block_sum(g1, sh);
    t3 = block_sum(g3, sh);
  }
  if (tid == 0) {
    const double v[5] = {t0, sc * t1 / s.P, sc * t2, sc * t1 / s.eta, sc * t3};
    for (int q = 0; q < 5; ++q) slot[q] = first ? (float)v[q] : (float)(slot[q] + v[q]);
  }
}

// The same in FP64 for finite differences, every voxel-step evaluated: loss only, 16x16x4 tiles,
// two row tiles per wave.
constexpr int KP64 = 28, CT64 = 16;
static __global__ __launch_bounds__(HB, 2) void k_heat64(Geo g, const Src* S, const Src* Tg, int step0, int nsteps, int ctiles,
                                               double* part, int first) {
  __shared__ double sG[2][2][KP64 * CT64];
  __shared__ double nk[2][4][KP64];  // per set: vtau, 1/D1, 1/(4 alpha tau), amp
  __shared__ double sh[HB / 64];
  const int lane = threadIdx.x, w = threadIdx.y, tid = 64 * w + lane;
  const Src s[2] = {S[blockIdx.z], Tg[blockIdx.z]};
  const int nyz = g.ny * g.nz;
  const long long ncol = (long long)nsteps * g.nx;
  const int ntile = (int)((ncol + CT64 - 1) / CT64);
  const int c0 = blockIdx.y * ctiles, c1 = min(ntile, c0 + ctiles);
  if (tid < KP64)
    for (int u = 0; u < 2; ++u) {
      const bool in = tid < NQ;
      const double tau = in ? g.h * (1 - kHx[tid]) : 1.0, W = in ? g.h * kHw[tid] : 0.0;
      const double C = s[u].eta * s[u].P / (M_PI * (g.k / g.alpha) * sqrt(4 * M_PI * g.alpha));
      const double A = 2 * g.alpha * tau + s[u].sigma * s[u].sigma;
      nk[u][0][tid] = in ? s[u].v * tau : 0.0;
      nk[u][1][tid] = in ? 1 / (2 * A) : 0.0;
      nk[u][2][tid] = in ? 1 / (4 * g.alpha * tau) : 0.0;
      nk[u][3][tid] = in ? W * C / (sqrt(tau) * A) : 0.0;
    }
  __syncthreads();
  double a[2][2][KP64 / 4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row = blockIdx.x * ROWS + w * RT + 16 * h + (lane & 15);
    const bool in = row < nyz;
    const int z = row / g.ny, y = row - z * g.ny;
    const double dy = (y + 0.5) * g.dx - g.ys, dz = (z + 0.5) * g.dx - g.zs;
#pragma unroll
    for (int p = 0; p < KP64 / 4; ++p) {
      const int q = 4 * p + (lane >> 4);
#pragma unroll
      for (int u = 0; u < 2; ++u)
        a[u][h][p] = in ? nk[u][3][q] * exp(-(dy * dy) * nk[u][1][q] - (dz * dz) * nk[u][2][q]) : 0.0;
    }
  }
  auto columns = [&](int tile, int buf) {
    const int c = tid & 15;
    const long long col = (long long)tile * CT64 + c;
    const bool in = col < ncol;
    const int m = in ? (int)(col / g.nx) : 0, i = in ? (int)(col - (long long)m * g.nx) : 0;
    const double t = (step0 + 1 + m) * g.dt, x0 = (i + 0.5) * g.dx - g.xs;
    for (int q = tid >> 4; q < KP64; q += HB / 16)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const double d = x0 - s[u].v * t + nk[u][0][q];
        sG[buf][u][q * CT64 + c] = in ? exp(-d * d * nk[u][1][q]) : 0.0;
      }
  };
  double loss = 0;
  const double iw = 1 / g.width;
  if (c0 < c1) columns(c0, 0);
  for (int tile = c0, buf = 0; tile < c1; ++tile, buf ^= 1) {
    __syncthreads();
    if (tile + 1 < c1) columns(tile + 1, buf ^ 1);
    f64x4 x[2][2] = {};
#pragma unroll
    for (int p = 0; p < KP64 / 4; ++p)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const double b = sG[buf][u][p * 64 + lane];
#pragma unroll
        for (int h = 0; h < 2; ++h) x[u][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][h][p], b, x[u][h], 0, 0, 0);
      }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double df = 1 / (1 + exp(-(x[0][h][r] + (g.T0 - g.tL)) * iw)) -
                          1 / (1 + exp(-(x[1][h][r] + (g.T0 - g.tL)) * iw));
        loss += df * df;
      }
  }
  const double t0 = block_sum(loss, sh);
  double* slot = part + 5 * ((size_t)(blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x);
  if (tid == 0) {
    slot[0] = first ? t0 : slot[0] + t0;
    if (first)
      for (int q = 1; q < 5; ++q) slot[q] = 0;
  }
}

// Sum of the block slots of each instance (blockIdx.x) in a fixed order: thread t adds
// slots t, t + 256, ... in order, then the 256 partial sums are added pairwise; in FP64.
template <typename F>
__global__ __launch_bounds__(256) void k_heat_reduce(const F* part, int nblk, F* out) {
  __shared__ double sh[256];
  const F* p = part + 5 * (size_t)blockIdx.x * nblk;
  double acc[5] = {0, 0, 0, 0, 0};
  for (int b = threadIdx.x; b < nblk; b += 256)
    for (int q = 0; q < 5; ++q) acc[q] += p[5 * (size_t)b + q];
  for (int q = 0; q < 5; ++q) {
    sh[threadIdx.x] = acc[q];
    __syncthreads();
    for (int w = 128; w >= 1; w >>= 1) {
      if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
      __syncthreads();
    }
    if (threadIdx.x == 0) out[5 * blockIdx.x + q] = (F)sh[0];
    __syncthreads();
  }
}

static inline Geo geo(const amcafe_heat_desc* d) {
  return {d->nX[0],    d->nX[1], d->nX[2], d->dX,    d->x_start, d->y_track, d->z_track,    d->dt,
          d->T0,       d->tL,    d->width, d->k,     d->alpha,   d->t_hist / 2};
}

#define HCHECK(x)                                                          \
  do {                                                                     \
    hipError_t e_ = (x);                                                   \
    if (e_ != hipSuccess) {                                                \
      snprintf(err, errlen, "%s: %s", #x, hipGetErrorString(e_));          \
      return -1;                                                           \
    }                                                                      \
  } while (0)

// Device buffers of one call: source parameters (theta then target, nb each), the block
// slots (5 values per block and instance), the per-instance sums and the evaluation counter.
template <typename F>
struct Bufs {
  Src* src;
  F* part;
  F* out;
  unsigned long long* evals;
};

// The launch shape of a call: segments of at most `checkpoint` steps and no longer than the call (nor than
// 2^30 columns, so that every count of tiles fits an int), groups of ROWS rows, and shares of `per` column
// tiles (FP32: 16, so few that the hot tenth of a 256x256x64 domain's 6400 blocks fills the chip; a
// cold block leaves after its bounds.  Loss / loss and gradient / 32 sets of 128x128x48, ms: 4 tiles
// 3.22 / 4.34 / 10.2, 8: 3.16 / 4.29 / 9.8, 16: 2.91 / 4.01 / 8.8, 32: 3.32 / 4.48 / 8.7; blocks of 128
// threads 3.13 / 4.58 / 9.4, of 512 3.6 / 5.8 / 12.8), and no more blocks than there are 256 voxels (the allocation-free
// call's account) unless there are more groups than that (nx = 1: at most twice).  Rows in patches of 8 x 4
// where the patches' padding is at most 1.9 times the rows and nx makes up for it.
struct Shape {
  int groups, runs, seg, patch, nx, ct;
  // column tiles of each share in a launch of `steps` steps: a segment shorter than the others is
  // spread over all shares too
  int ctiles(int steps) const {
    const long long tiles = ((long long)steps * nx + ct - 1) / ct;
    return (int)((tiles + runs - 1) / runs);
  }
};
static inline Shape shape(const amcafe_heat_desc* d, int nsteps, int ct, int per, bool patches) {
  Shape s;
  const int nx = d->nX[0], ny = d->nX[1], nz = d->nX[2];
  s.nx = nx;
  s.ct = ct;
  s.seg = std::min({d->checkpoint > 0 ? d->checkpoint : 100, std::max(nsteps, 1), std::max((1 << 30) / nx, 1)});
  s.patch = patches && nx >= 2 && ny >= 16 && nz >= 8;
  const long long rtiles = s.patch ? (long long)((ny + 7) / 8) * ((nz + 3) / 4) : ((long long)ny * nz + RT - 1) / RT;
  s.groups = (int)((rtiles + HB / 64 - 1) / (HB / 64));
  const long long tiles = ((long long)s.seg * nx + ct - 1) / ct;
  const long long blocks = ((long long)nx * ny * nz + 255) / 256;
  const long long runs = std::max<long long>(1, std::min<long long>({(tiles + per - 1) / per, blocks / s.groups, 65535}));
  const long long share = (tiles + runs - 1) / runs;
  s.runs = (int)((tiles + share - 1) / share);
  return s;
}
template <typename F>
static Shape shape_of(const amcafe_heat_desc* d, int nsteps) {
  return sizeof(F) == 8 ? shape(d, nsteps, CT64, 8, false) : shape(d, nsteps, CT, 16, true);
}

// The call's segments, one launch each (all instances of the batch in it),
// then the fixed-order reduction; everything on `stream`.  No steps: every slot holds zero.
template <typename F, bool GRAD>
static void launch_all(const amcafe_heat_desc* d, int nb, const Bufs<F>& B, int step0, int nsteps,
                       hipStream_t stream) {
  const Shape h = shape_of<F>(d, nsteps);
  const Geo g = geo(d);
  // (64 threads along x: a launch counts its threads in 32 bits per dimension, and there may be 2^24 groups)
  const dim3 grid(h.groups, h.runs, nb), block(64, HB / 64);
  for (long long m = 0; m == 0 || m < nsteps; m += h.seg) {
    const int c = (int)std::max(0ll, std::min<long long>(nsteps - m, h.seg)), ctiles = h.ctiles(c);
    if constexpr (sizeof(F) == 8)
      hipLaunchKernelGGL(k_heat64, grid, block, 0, stream, g, B.src, B.src + nb, (int)(step0 + m), c, ctiles, B.part,
                         m == 0 ? 1 : 0);
    else
      hipLaunchKernelGGL((k_heat<GRAD>), grid, block, 0, stream, g, B.src, B.src + nb, (int)(step0 + m), c, ctiles,
                         h.patch, B.part, m == 0 ? 1 : 0, B.evals);
  }
  hipLaunchKernelGGL((k_heat_reduce<F>), dim3(nb), dim3(256), 0, stream, B.part, h.groups * h.runs, B.out);
}

static inline void sources(int nb, const double* theta, const double* target, std::vector<Src>& hs) {
  hs.resize(2 * (size_t)nb);
  for (int b = 0; b < nb; ++b) {
    hs[b] = {theta[4 * b], theta[4 * b + 1], theta[4 * b + 2], theta[4 * b + 3]};
    hs[nb + b] = {target[4 * b], target[4 * b + 1], target[4 * b + 2], target[4 * b + 3]};
  }
}

template <typename F>
static void results(int nb, const std::vector<F>& h, bool grad_on, double* loss, double* grad) {
  for (int b = 0; b < nb; ++b) {
    if (loss) loss[b] = (double)h[5 * b];
    if (grad_on && grad)
      for (int q = 0; q < 4; ++q) grad[4 * b + q] = (double)h[5 * b + 1 + q];
  }
}

}  // namespace amcafe_heat
