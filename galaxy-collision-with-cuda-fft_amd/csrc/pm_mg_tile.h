// One launch per leg of a V-cycle on the coarse levels: the down leg smooths, evaluates the
// residual and restricts it; the up leg prolongs, corrects and smooths.
//
// The levels below the finest are small (a 129^3 level is 8.6 MB an array, a 65^3 one 1.1 MB):
// their colour passes, residuals, restrictions and prolongations run from the caches and each
// launch costs its few microseconds of latency whatever it does. A leg therefore gives every
// workgroup an 8^3 block of nodes and enough nodes around it (two per sweep, one for the
// residual, one for the restriction) to run the whole leg in LDS: nodes near the region's edge
// turn stale one layer a colour pass and never reach the block. Each node is updated with the
// expressions of the per-pass kernels in their order from the same inputs, so every value is
// bitwise theirs, wherever it is computed.
//
// Blocks cover the interior nodes 1 .. n-2 (block b the nodes 8b+1 .. 8b+8 of an axis, which
// hold the coarse nodes 4b+1 .. 4b+4), so an aligned 2^m + 1 level wastes no block on faces.
// The region lies in LDS in natural order, so a node's neighbours are at constant offsets; a
// pass gives each lane the same (j, k) in every few planes, so a step costs no index
// arithmetic, and it covers only the layers that are still needed.
//
// Bound: the region's passes on one CU (a colour pass of a 17^3 region takes about 1.2 us, LDS
// and issue) and, from 65^3 up, the nodes updated more than once (a block of 8^3 computes on
// up to 17^3). Measured per leg on the MI355X, us, against the per-pass kernels it replaces:
// 33^3 V(1,1) 4.8 down, 5.8 up (9.5, 7.5), V(2,2) 8.4, 9.8 (13, 12); 65^3 V(1,1) 6.2, 6.9
// (9.9, 8.3), V(2,2) 11.7, 13.3 (14.7, 13.0). At 129^3 V(2,2) the leg takes 60 and 73 us against 39 and 40, and 16^3
// blocks 41 and 41: levels above kLegMax keep a launch per pass. 4^3 blocks measured 4.0 and 4.2 us at
// 33^3 V(1,1) but 8.4 and 9.1 at V(2,2) and lost from 41^3 up.
#pragma once

#include <hip/hip_runtime.h>

#include "pm_common.h"

namespace pm {
namespace tile {

constexpr int K = 8;    // nodes of a block per axis
constexpr int T = 512;  // threads of a workgroup

// x[m] / 6 rounded once, for M values: the quotient by the rounded reciprocal corrected with
// its exact remainder (Markstein) equals the IEEE division where nothing under- or overflows
// (checked for every mantissa; a zero keeps its sign by the copysign). A wave that holds any
// other argument repeats its values by division: one branch for all of them, so that the M
// chains overlap.
template <int M>
__device__ __forceinline__ void div6(float (&x)[M]) {
  constexpr float r = 0x1.555556p-3f;
  float out[M];
  bool ok = true;
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const float a = __builtin_fabsf(x[m]);
    const float q = x[m] * r;
    out[m] = __builtin_copysignf(__builtin_fmaf(__builtin_fmaf(-6.0f, q, x[m]), r, q), x[m]);
    ok = ok && (a == 0.0f || (a >= 0x1p-100f && a <= 0x1p100f));
  }
  if (!ok) {
#pragma unroll
    for (int m = 0; m < M; ++m) out[m] = x[m] / 6.0f;
  }
#pragma unroll
  for (int m = 0; m < M; ++m) x[m] = out[m];
}

// What a region needs to know of the grid: its origin, and whether it reaches past the interior
// nodes (uniform over the workgroup: only such regions test their nodes).
struct Place {
  int n, i0, j0, k0;
  bool edge;
  __device__ __forceinline__ bool inner(int a, int b, int c) const {
    const int i = i0 + a, j = j0 + b, k = k0 + c;
    return i >= 1 && i <= n - 2 && j >= 1 && j <= n - 2 && k >= 1 && k <= n - 2;
  }
};

// Flat index of node (i, j, k), n <= 1024: 32 bits hold it and 24-bit products form it (a full
// 32-bit product takes four times as long).
__device__ __forceinline__ uint32_t node(int i, int j, int k, int n) {
  const uint32_t row = __umul24(static_cast<uint32_t>(i), static_cast<uint32_t>(n)) +
                       static_cast<uint32_t>(j);
  return __umul24(row, static_cast<uint32_t>(n)) + static_cast<uint32_t>(k);
}

// t / D for 0 <= t < 2^14 and 5 <= D < 64 by one 24-bit product: the multiplier exceeds
// 2^20 / D by at most 1, so the quotient's excess stays below 2^14 / 2^20 = 1 / 64.
template <int D>
__device__ __forceinline__ int div_c(int t) {
  static_assert(D >= 5 && D < 64, "divisor range");
  return static_cast<int>(__umul24(static_cast<uint32_t>(t), (1u << 20) / D + 1u) >> 20);
}

// (a, b, c) of region-ordered index t on an S^3 box.
template <int S>
__device__ __forceinline__ void split3(int t, int& a, int& b, int& c) {
  const int q = div_c<S>(t);
  c = t - q * S;
  a = div_c<S>(q);
  b = q - a * S;
}

// Region of workgroup w in an nb^3 arrangement of K^3 blocks with D nodes before each block.
template <int D, int R>
__device__ __forceinline__ Place place(int n, int nb, int& bi, int& bj, int& bk) {
  const uint32_t w = static_cast<uint32_t>(pm::xcd_block()), u = static_cast<uint32_t>(nb);
  bk = static_cast<int>(w % u);
  bj = static_cast<int>((w / u) % u);
  bi = static_cast<int>(w / (u * u));
  Place p;
  p.n = n;
  p.i0 = K * bi + 1 - D;
  p.j0 = K * bj + 1 - D;
  p.k0 = K * bk + 1 - D;
  p.edge = p.i0 < 1 || p.j0 < 1 || p.k0 < 1 || p.i0 + R - 1 > n - 2 || p.j0 + R - 1 > n - 2 ||
           p.k0 + R - 1 > n - 2;
  return p;
}

// Sum of a node's six neighbours in rb_pass_kernel's order.
template <int R>
__device__ __forceinline__ float nbr_sum(const float* p) {
  return p[R * R] + p[-R * R] + p[R] + p[-R] + p[1] + p[-1];
}

// One colour pass over the region's layers L and deeper. PAR: colour of region node (0, 0, 0).
// A pass reads only the other colour, so every new value is formed before the first is stored.
template <int R, int L, int COLOR, int PAR>
__device__ __forceinline__ void colour_pass(float* phi, const float* rhs, const Place& pl,
                                            float h2) {
  constexpr int W = R - 2 * L, HW = (W + 1) / 2, kLanes = W * HW;
  static_assert(kLanes <= T, "a plane's nodes of one colour fit the workgroup");
  constexpr int kPlanes = T / kLanes >= 2 ? (T / kLanes) / 2 * 2 : 1;  // planes a step
  constexpr int kSteps = (W + kPlanes - 1) / kPlanes;
  const int t = static_cast<int>(threadIdx.x);
  const int q = t / kLanes, rem = t - q * kLanes, bb = rem / HW;
  const int a0 = L + q, b = L + bb, c0 = L + 2 * (rem - bb * HW);
  const int f = (a0 + b + L + PAR + COLOR) & 1;
  // kGroup steps at a time: their loads are issued before any is used (from a safe node where
  // the lane has none), and their divisions overlap
  constexpr int kSafe = (R + 1) * R + 1;
  constexpr int kGroup = 4;
#pragma unroll
  for (int s0 = 0; s0 < kSteps; s0 += kGroup) {
    float out[kGroup];
    int o[kGroup];
#pragma unroll
    for (int g = 0; g < kGroup; ++g) {
      const int st = s0 + g, a = a0 + st * kPlanes;
      const int c = c0 + (kPlanes == 1 ? f ^ (st & 1) : f);
      const bool on = st < kSteps && q < kPlanes && a <= R - 1 - L && c <= R - 1 - L &&
                      (!pl.edge || pl.inner(a, b, c));
      o[g] = on ? (a * R + b) * R + c : -1;
      const int from = on ? o[g] : kSafe;
      out[g] = nbr_sum<R>(phi + from) - h2 * rhs[from];
    }
    div6<kGroup>(out);
#pragma unroll
    for (int g = 0; g < kGroup; ++g)
      if (o[g] >= 0) phi[o[g]] = out[g];
  }
  __syncthreads();
}

// The colour passes of NU sweeps; pass p (from 1) is valid from layer p (minus 1 where the
// first colour-0 pass, done at the load, needed no neighbours).
template <int R, int NU, bool ZERO, int PAR>
__device__ __forceinline__ void smooth(float* phi, const float* rhs, const Place& pl, float h2) {
  constexpr int z = ZERO ? 1 : 0;
  if constexpr (!ZERO) colour_pass<R, 1, 0, PAR>(phi, rhs, pl, h2);
  colour_pass<R, 2 - z, 1, PAR>(phi, rhs, pl, h2);
  if constexpr (NU == 2) {
    colour_pass<R, 3 - z, 0, PAR>(phi, rhs, pl, h2);
    colour_pass<R, 4 - z, 1, PAR>(phi, rhs, pl, h2);
  }
}

inline int blocks_per_axis(int n) { return (n - 2 + K - 1) / K; }

// Down leg: phi_out = NU sweeps from zero, interior nodes only; rhs_c = full weighting of
// rhs - lap(phi_out) and phi_c = 0 on the coarse interior.
template <int NU>
__global__ void __launch_bounds__(T) down_kernel(const float* __restrict__ rhs,
                                                 float* __restrict__ phi_out,
                                                 float* __restrict__ rhs_c,
                                                 float* __restrict__ phi_c, int n, int nc, int nb,
                                                 float h2, float inv_h2) {
  constexpr int D = 2 * NU;      // region coordinate of the block's first node
  constexpr int R = K + 1 + 2 * D;
  constexpr int W = K + 1;       // residual nodes per axis
  constexpr int PAR = (1 - D) & 1;  // K is even, so every region has the same parity
  constexpr int N = R * R * R;
  __shared__ float s[N];
  __shared__ float sr[N];
  __shared__ float res[W * W * W];
  int bi, bj, bk;
  const Place pl = place<D, R>(n, nb, bi, bj, bk);
  constexpr int kLoads = (N + T - 1) / T;
  {
    float rv[kLoads];
#pragma unroll
    for (int m = 0; m < kLoads; ++m) {
      const int t = static_cast<int>(threadIdx.x) + m * T;
      int a, b, c;
      split3<R>(t, a, b, c);
      const int i = pl.i0 + a, j = pl.j0 + b, k = pl.k0 + c;
      const bool ok = t < N && (!pl.edge || (i >= 0 && i < n && j >= 0 && j < n && k >= 0 && k < n));
      const uint32_t o = ok ? node(i, j, k, n) : 0u;
      rv[m] = rhs[o];
      rv[m] = ok ? rv[m] : 0.0f;
    }
    // the first colour-0 pass from a zero guess reads no neighbour (their sum is +0)
    constexpr int kBatch = 4;
#pragma unroll
    for (int m0 = 0; m0 < kLoads; m0 += kBatch) {
      float e[kBatch];
#pragma unroll
      for (int g = 0; g < kBatch; ++g)
        e[g] = 0.0f - h2 * (m0 + g < kLoads ? rv[m0 + g] : 0.0f);
      div6<kBatch>(e);
#pragma unroll
      for (int g = 0; g < kBatch; ++g) {
        const int t = static_cast<int>(threadIdx.x) + (m0 + g) * T;
        if (m0 + g >= kLoads || t >= N) continue;
        int a, b, c;
        split3<R>(t, a, b, c);
        const bool red = ((a + b + c + PAR) & 1) == 0 && (!pl.edge || pl.inner(a, b, c));
        s[t] = red ? e[g] : 0.0f;
        sr[t] = rv[m0 + g];
      }
    }
  }
  __syncthreads();
  smooth<R, NU, true, PAR>(s, sr, pl, h2);
  constexpr int kRes = (W * W * W + T - 1) / T;
  {
    float own[kRes], val[kRes];
#pragma unroll
    for (int m = 0; m < kRes; ++m) {
      const int t = min(static_cast<int>(threadIdx.x) + m * T, W * W * W - 1);
      int a, b, c;
      split3<W>(t, a, b, c);
      const int o = ((a + D) * R + (b + D)) * R + (c + D);
      own[m] = s[o];
      const float lap = (nbr_sum<R>(s + o) - 6.0f * own[m]) * inv_h2;
      // the residual of a face is 0
      val[m] = (!pl.edge || pl.inner(a + D, b + D, c + D)) ? sr[o] - lap : 0.0f;
    }
#pragma unroll
    for (int m = 0; m < kRes; ++m) {
      const int t = static_cast<int>(threadIdx.x) + m * T;
      if (t >= W * W * W) continue;
      res[t] = val[m];
      int a, b, c;
      split3<W>(t, a, b, c);
      if (a < K && b < K && c < K && (!pl.edge || pl.inner(a + D, b + D, c + D)))
        phi_out[node(pl.i0 + a + D, pl.j0 + b + D, pl.k0 + c + D, n)] = own[m];
    }
  }
  __syncthreads();
  constexpr int C = K / 2;
  if (threadIdx.x < C * C * C) {
    const int kc = threadIdx.x % C, jc = (threadIdx.x / C) % C, ic = threadIdx.x / (C * C);
    const int I = C * bi + 1 + ic, J = C * bj + 1 + jc, Kc = C * bk + 1 + kc;
    if (I <= nc - 2 && J <= nc - 2 && Kc <= nc - 2) {
      float acc = 0.0f;
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 3; ++b)
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const float w = (a == 1 ? 2.0f : 1.0f) * (b == 1 ? 2.0f : 1.0f) * (d == 1 ? 2.0f : 1.0f);
            acc += w * res[((2 * ic + a) * W + (2 * jc + b)) * W + (2 * kc + d)];
          }
      const uint32_t o = node(I, J, Kc, nc);
      rhs_c[o] = acc / 64.0f;
      phi_c[o] = 0.0f;
    }
  }
}

// Up leg: phi = NU sweeps from phi_in + prolongation(phi_c), interior nodes only; faces are
// read from phi (phi_in holds interior nodes, as the down leg leaves them).
template <int NU>
__global__ void __launch_bounds__(T) up_kernel(const float* __restrict__ phi_in,
                                               const float* __restrict__ rhs,
                                               const float* __restrict__ phi_c, float* phi, int n,
                                               int nc, int nb, float h2) {
  constexpr int D = 2 * NU;
  constexpr int R = K + 2 * D;
  constexpr int W = R / 2 + 2;  // coarse nodes per axis
  constexpr int PAR = (1 - D) & 1;
  constexpr int N = R * R * R;
  __shared__ float s[N];
  __shared__ float sr[N];
  __shared__ float cs[W * W * W];
  int bi, bj, bk;
  const Place pl = place<D, R>(n, nb, bi, bj, bk);
  // coarse nodes under the region (the origin may be negative: arithmetic shifts)
  const int ci0 = pl.i0 >> 1, cj0 = pl.j0 >> 1, ck0 = pl.k0 >> 1;
  constexpr int kCoarse = (W * W * W + T - 1) / T;
  constexpr int kLoads = (N + T - 1) / T;
  float cv[kCoarse], rv[kLoads], pv[kLoads];
#pragma unroll
  for (int m = 0; m < kCoarse; ++m) {
    const int t = static_cast<int>(threadIdx.x) + m * T;
    int a, b, c;
    split3<W>(t, a, b, c);
    const int ic = ci0 + a, jc = cj0 + b, kc = ck0 + c;
    const bool ok = t < W * W * W && ic >= 0 && ic < nc && jc >= 0 && jc < nc && kc >= 0 && kc < nc;
    cv[m] = phi_c[ok ? node(ic, jc, kc, nc) : 0u];
    cv[m] = ok ? cv[m] : 0.0f;
  }
#pragma unroll
  for (int m = 0; m < kLoads; ++m) {
    const int t = static_cast<int>(threadIdx.x) + m * T;
    int a, b, c;
    split3<R>(t, a, b, c);
    const int i = pl.i0 + a, j = pl.j0 + b, k = pl.k0 + c;
    const bool on = t < N && (!pl.edge || (i >= 0 && i < n && j >= 0 && j < n && k >= 0 && k < n));
    const bool in = on && (!pl.edge || pl.inner(a, b, c));
    const uint32_t o = on ? node(i, j, k, n) : 0u;
    rv[m] = rhs[o];
    pv[m] = phi_in[o];
    if (pl.edge && on && !in) pv[m] = phi[o];
    rv[m] = in ? rv[m] : 0.0f;
    pv[m] = on ? pv[m] : 0.0f;
  }
#pragma unroll
  for (int m = 0; m < kCoarse; ++m) {
    const int t = static_cast<int>(threadIdx.x) + m * T;
    if (t < W * W * W) cs[t] = cv[m];
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < kLoads; ++m) {
    const int t = static_cast<int>(threadIdx.x) + m * T;
    if (t >= N) continue;
    int a, b, c;
    split3<R>(t, a, b, c);
    // the origin is odd on every axis (D is even), so region parities give the grid's
    const int oi = (a & 1) ^ 1, oj = (b & 1) ^ 1, ok = (c & 1) ^ 1;
    const float* p = cs + (((a + 1) >> 1) * W + ((b + 1) >> 1)) * W + ((c + 1) >> 1);
    // prolong_value's sum: terms of weight 0 are not added
    float val = 0.0f;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int di = u >> 2, dj = (u >> 1) & 1, dk = u & 1;
      const float w = (oi ? 0.5f : (di == 0 ? 1.0f : 0.0f)) * (oj ? 0.5f : (dj == 0 ? 1.0f : 0.0f)) *
                      (ok ? 0.5f : (dk == 0 ? 1.0f : 0.0f));
      const float v = val + w * p[(di * W + dj) * W + dk];
      val = w > 0.0f ? v : val;
    }
    const float out = (!pl.edge || pl.inner(a, b, c)) ? pv[m] + val : pv[m];
    s[t] = out;
    sr[t] = rv[m];
  }
  __syncthreads();
  smooth<R, NU, false, PAR>(s, sr, pl, h2);
  constexpr int kOut = (K * K * K + T - 1) / T;
#pragma unroll
  for (int m = 0; m < kOut; ++m) {
    const int t = static_cast<int>(threadIdx.x) + m * T;
    if (t >= K * K * K) continue;
    const int c = t % K, b = (t / K) % K, a = t / (K * K);
    if (pl.edge && !pl.inner(a + D, b + D, c + D)) continue;
    phi[node(pl.i0 + a + D, pl.j0 + b + D, pl.k0 + c + D, n)] =
        s[((a + D) * R + (b + D)) * R + (c + D)];
  }
}

}  // namespace tile
}  // namespace pm
