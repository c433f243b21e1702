// Warm-start kernels of the multigrid solve: linear extrapolation of phi in time, the
// learned correction's input (pooled, normalized fine fields) and output (trilinear
// interpolation onto the fine grid), the residual check that judges it, and the training
// target written after a solve.
//
// Coarse voxel V = (Z, Y, X) of the network grid (R = n / p per axis) covers the fine nodes
// p*V .. p*V + p-1 along each axis; its value is their mean. The fine node i sits at coarse
// coordinate u = (i - (p-1)/2) / p, so interpolation back is the cell-centred trilinear
// rule with edge clamping.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "pm_common.h"
#include "pm_conv.h"
#include "pm_reduce.h"
#include "pm_timing.h"
#include "pm_warm.h"

namespace {

using pm::conv::f2bf;

// phi_new = 2*phi - hist on the interior (faces keep phi's values); hist = phi (old) on
// every node; cand = phi_new if requested.
__global__ void __launch_bounds__(256) extrap_kernel(float* __restrict__ phi,
                                                     float* __restrict__ hist,
                                                     float* __restrict__ cand, int n) {
  const int64_t c = pm::xcd_block() * blockDim.x + threadIdx.x;
  const int64_t total = static_cast<int64_t>(n) * n * n;
  if (c >= total) return;
  const pm::Idx3 q = pm::idx3(c, n);
  const float p = phi[c];
  float v = p;
  if (q.i >= 1 && q.i <= n - 2 && q.j >= 1 && q.j <= n - 2 && q.k >= 1 && q.k <= n - 2)
    v = 2.0f * p - hist[c];
  phi[c] = v;
  hist[c] = p;
  if (cand) cand[c] = v;
}

// extrap_kernel, 4 nodes of a row per thread (n % 4 == 0, 16-byte aligned arrays). Memory
// bound: 45 us at 256^3 (268 MB), where one node per thread, also writing cand, took 89.
__global__ void __launch_bounds__(256) extrap4_kernel(float* __restrict__ phi,
                                                      float* __restrict__ hist,
                                                      float* __restrict__ cand, int n) {
  const int64_t t = pm::xcd_block() * blockDim.x + threadIdx.x;
  const int64_t total = static_cast<int64_t>(n) * n * n;
  if (4 * t >= total) return;
  const pm::Idx3 q = pm::idx3(4 * t, n);
  const float4 p = reinterpret_cast<const float4*>(phi)[t];
  const float4 h = reinterpret_cast<const float4*>(hist)[t];
  const bool inner = q.i >= 1 && q.i <= n - 2 && q.j >= 1 && q.j <= n - 2;
  float4 v;
  v.x = inner && q.k >= 1 ? 2.0f * p.x - h.x : p.x;
  v.y = inner ? 2.0f * p.y - h.y : p.y;
  v.z = inner ? 2.0f * p.z - h.z : p.z;
  v.w = inner && q.k + 3 <= n - 2 ? 2.0f * p.w - h.w : p.w;
  reinterpret_cast<float4*>(phi)[t] = v;
  reinterpret_cast<float4*>(hist)[t] = p;
  if (cand) reinterpret_cast<float4*>(cand)[t] = v;
}

// Slab decomposition shared by the kernels below: slab (Z, Y, seg) is the p x p x 64 block
// of fine nodes i = p*Z + a, j = p*Y + b, k = 64*seg + lane (a, b < p), i.e. the fine nodes
// of 64/p consecutive network voxels along x. Lane = k offset (coalesced rows), wave w takes
// the (a, b) pairs w, w+4, ...; p divides 64.
constexpr int kSeg = 64;

struct Slab {
  int Z, Y, seg;
};

__device__ __forceinline__ Slab slab_of(int64_t slab, int R, int nseg) {
  // (at most 1024^2 * 16 slabs: 32-bit divisions)
  const uint32_t t = static_cast<uint32_t>(slab), row = t / static_cast<uint32_t>(nseg);
  Slab q;
  q.seg = static_cast<int>(t - row * static_cast<uint32_t>(nseg));
  q.Z = static_cast<int>(row / static_cast<uint32_t>(R));
  q.Y = static_cast<int>(row - static_cast<uint32_t>(q.Z) * static_cast<uint32_t>(R));
  return q;
}

// Sums Q per-thread values over the block's 4 waves (LDS) and then over aligned groups of p
// lanes (shuffles): on return lane X*p of wave 0 holds the sum over the p^3 fine nodes of
// network voxel X of the slab. Contains __syncthreads(): uniform control flow only.
template <int Q>
__device__ __forceinline__ void slab_reduce(float (&t)[Q], int p, float (*s)[kSeg][Q]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < Q; ++q) s[wave][lane][q] = t[q];
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int q = 0; q < Q; ++q) t[q] = ((s[0][lane][q] + s[1][lane][q]) + s[2][lane][q]) + s[3][lane][q];
    for (int off = 1; off < p; off <<= 1) {
#pragma unroll
      for (int q = 0; q < Q; ++q) t[q] += __shfl_down(t[q], off, 64);
    }
  }
  __syncthreads();
}

// Pooled channels [r, phi - hist, f = factor*rho] of every network voxel -> pooled[V][3]; float64
// partial sums of their squares (grid-stride over slabs, fixed order per launch size).
__global__ void __launch_bounds__(256) pool_input_kernel(const float* __restrict__ r32,
                                                         const float* __restrict__ phi,
                                                         const float* __restrict__ hist,
                                                         const float* __restrict__ rho,
                                                         float factor, int n, int p, int R,
                                                         float* __restrict__ pooled,
                                                         double* __restrict__ partials) {
  __shared__ float s[4][kSeg][3];
  __shared__ double s_red[4 * 3];
  double v[3] = {0.0, 0.0, 0.0};
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nseg = (n + kSeg - 1) / kSeg;
  const int64_t slabs = static_cast<int64_t>(R) * R * nseg;
  const float inv = 1.0f / static_cast<float>(p * p * p);
  for (int64_t sl = blockIdx.x; sl < slabs; sl += gridDim.x) {
    const Slab q = slab_of(sl, R, nseg);
    const int k = q.seg * kSeg + lane;
    float t[3] = {0.0f, 0.0f, 0.0f};
    if (k < n) {
      for (int ab = wave; ab < p * p; ab += 4) {
        const int i = p * q.Z + ab / p, j = p * q.Y + ab % p;
        const int64_t c = (static_cast<int64_t>(i) * n + j) * n + k;
        t[0] += r32[c];
        t[1] += phi[c] - hist[c];
        t[2] += factor * rho[c];
      }
    }
    slab_reduce<3>(t, p, s);
    if (wave == 0 && k < n && lane % p == 0) {
      const int64_t V = (static_cast<int64_t>(q.Z) * R + q.Y) * R + k / p;
      for (int c = 0; c < 3; ++c) {
        const float o = t[c] * inv;
        pooled[V * 3 + c] = o;
        v[c] = v[c] + static_cast<double>(o) * static_cast<double>(o);
      }
    }
  }
  pm::block_sum<3>(v, s_red);
  if (threadIdx.x == 0)
    for (int c = 0; c < 3; ++c) partials[blockIdx.x * pm::kRedMaxQ + c] = v[c];
}

// scales[q] = RMS of pooled channel q (q < 3); scales[3] = RMS(r) * (p*h)^2, the output
// scale; scales[4] = 1 / scales[3] (0 when the residual vanishes).
__global__ void scales_kernel(const double* __restrict__ sums, int64_t nv, double ph2,
                              float* __restrict__ scales) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  for (int q = 0; q < 3; ++q) scales[q] = static_cast<float>(std::sqrt(sums[q] / nv));
  const double so = std::sqrt(sums[0] / nv) * ph2;
  scales[3] = static_cast<float>(so);
  scales[4] = so > 0.0 ? static_cast<float>(1.0 / so) : 0.0f;
}

// input[V][0..7] = bf16(pooled[V][q] / scales[q]) for q < 3, 0 for the pad channels.
__global__ void __launch_bounds__(256) normalize_kernel(const float* __restrict__ pooled,
                                                        int64_t nv,
                                                        const float* __restrict__ scales,
                                                        uint16_t* __restrict__ input) {
  const int64_t V = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (V >= nv) return;
  uint16_t h[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int q = 0; q < 3; ++q) {
    const float s = scales[q];
    h[q] = f2bf(s > 0.0f ? pooled[V * 3 + q] / s : 0.0f);
  }
  uint4 w;
  w.x = h[0] | (static_cast<uint32_t>(h[1]) << 16);
  w.y = h[2] | (static_cast<uint32_t>(h[3]) << 16);
  w.z = h[4] | (static_cast<uint32_t>(h[5]) << 16);
  w.w = h[6] | (static_cast<uint32_t>(h[7]) << 16);
  *reinterpret_cast<uint4*>(input + V * 8) = w;
}

__device__ __forceinline__ void interp_axis(int i, int p, int R, int& i0, int& i1, float& w) {
  // u = (i - (p-1)/2) / p: the node's coordinate in network voxels (cell centres)
  const float u = static_cast<float>(2 * i - (p - 1)) / static_cast<float>(2 * p);
  const float f = floorf(u);
  w = u - f;
  const int a = static_cast<int>(f);
  i0 = a < 0 ? 0 : (a > R - 1 ? R - 1 : a);
  i1 = a + 1 < 0 ? 0 : (a + 1 > R - 1 ? R - 1 : a + 1);
}

// The network's output at fine node (i, j, k): along x, then y, then z.
__device__ __forceinline__ float trilinear(const float* __restrict__ out, int R, int p, int i,
                                           int j, int k) {
  int x0, x1, y0, y1, z0, z1;
  float wx, wy, wz;
  interp_axis(k, p, R, x0, x1, wx);
  interp_axis(j, p, R, y0, y1, wy);
  interp_axis(i, p, R, z0, z1, wz);
  const float* r00 = out + (static_cast<int64_t>(z0) * R + y0) * R;
  const float* r01 = out + (static_cast<int64_t>(z0) * R + y1) * R;
  const float* r10 = out + (static_cast<int64_t>(z1) * R + y0) * R;
  const float* r11 = out + (static_cast<int64_t>(z1) * R + y1) * R;
  const float c00 = r00[x0] * (1.0f - wx) + r00[x1] * wx;
  const float c01 = r01[x0] * (1.0f - wx) + r01[x1] * wx;
  const float c10 = r10[x0] * (1.0f - wx) + r10[x1] * wx;
  const float c11 = r11[x0] * (1.0f - wx) + r11[x1] * wx;
  const float c0 = c00 * (1.0f - wy) + c01 * wy;
  const float c1 = c10 * (1.0f - wy) + c11 * wy;
  return c0 * (1.0f - wz) + c1 * wz;
}

// e = scales[3] * trilinear(out) on the interior, 0 on the faces; one slab per block.
__global__ void __launch_bounds__(256) apply_kernel(const float* __restrict__ out, int R, int p,
                                                    int n, const float* __restrict__ scales,
                                                    float* __restrict__ e) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nseg = (n + kSeg - 1) / kSeg;
  const Slab q = slab_of(blockIdx.x, R, nseg);
  const int k = q.seg * kSeg + lane;
  if (k >= n) return;  // no barriers below
  const float so = scales[3];
  for (int ab = wave; ab < p * p; ab += 4) {
    const int i = p * q.Z + ab / p, j = p * q.Y + ab % p;
    const int64_t c = (static_cast<int64_t>(i) * n + j) * n + k;
    float val = 0.0f;
    if (i >= 1 && i <= n - 2 && j >= 1 && j <= n - 2 && k >= 1 && k <= n - 2) {
      val = so * trilinear(out, R, p, i, j, k);
    }
    e[c] = val;
  }
}

// Place of node (i, j, k): natural order (hn = 0), or colour planes of rows of hn positions.
__device__ __forceinline__ int64_t place(int i, int j, int k, int n, int hn) {
  const int64_t row = static_cast<int64_t>(i) * n + j;
  if (hn == 0) return row * n + k;
  return ((i + j + k) & 1) * static_cast<int64_t>(n) * n * hn + row * hn + (k >> 1);
}

// The judge of a learned correction e. Per fine node: r' = r - lap(e) in float64 on the
// interior (0 on the faces), written to rnew (the residual of the corrected guess, colour-split
// with rows of hn positions when hn > 0); per
// network voxel: the mean residual before (r) and after (r'). Float64 partial sums of
// [mean before^2, mean after^2, r'^2]. The pooled residual measures the smooth error the
// correction targets (the full-resolution residual norm is dominated by high-frequency
// components that the smoother removes anyway).
__global__ void __launch_bounds__(256) guard_kernel(const float* __restrict__ r32,
                                                    const float* __restrict__ e, int n, int p,
                                                    int R, double inv_h2,
                                                    float* __restrict__ rnew, int hn,
                                                    double* __restrict__ partials) {
  __shared__ float s[4][kSeg][2];
  __shared__ double s_red[4 * 3];
  double v[3] = {0.0, 0.0, 0.0};
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nseg = (n + kSeg - 1) / kSeg;
  const int64_t slabs = static_cast<int64_t>(R) * R * nseg;
  const int64_t n2 = static_cast<int64_t>(n) * n;
  const float inv = 1.0f / static_cast<float>(p * p * p);
  for (int64_t sl = blockIdx.x; sl < slabs; sl += gridDim.x) {
    const Slab q = slab_of(sl, R, nseg);
    const int k = q.seg * kSeg + lane;
    float t[2] = {0.0f, 0.0f};
    if (k < n) {
      for (int ab = wave; ab < p * p; ab += 4) {
        const int i = p * q.Z + ab / p, j = p * q.Y + ab % p;
        const int64_t c = (static_cast<int64_t>(i) * n + j) * n + k;
        double ra = 0.0, rb = 0.0;
        if (i >= 1 && i <= n - 2 && j >= 1 && j <= n - 2 && k >= 1 && k <= n - 2) {
          const double sum = static_cast<double>(e[c + n2]) + static_cast<double>(e[c - n2]) +
                             static_cast<double>(e[c + n]) + static_cast<double>(e[c - n]) +
                             static_cast<double>(e[c + 1]) + static_cast<double>(e[c - 1]);
          rb = static_cast<double>(r32[c]);
          ra = rb - (sum - 6.0 * static_cast<double>(e[c])) * inv_h2;
        }
        rnew[place(i, j, k, n, hn)] = static_cast<float>(ra);
        v[2] = v[2] + ra * ra;
        t[0] += static_cast<float>(rb);
        t[1] += static_cast<float>(ra);
      }
    }
    slab_reduce<2>(t, p, s);
    if (wave == 0 && k < n && lane % p == 0) {
      const double mb = static_cast<double>(t[0] * inv), ma = static_cast<double>(t[1] * inv);
      v[0] = v[0] + mb * mb;
      v[1] = v[1] + ma * ma;
    }
  }
  pm::block_sum<3>(v, s_red);
  if (threadIdx.x == 0)
    for (int c = 0; c < 3; ++c) partials[blockIdx.x * pm::kRedMaxQ + c] = v[c];
}

// phi += e (0 on the faces)
__global__ void __launch_bounds__(256) add_kernel(float* __restrict__ phi,
                                                  const float* __restrict__ e, int64_t count) {
  const int64_t c = pm::xcd_block() * blockDim.x + threadIdx.x;
  if (c < count) phi[c] = phi[c] + e[c];
}

// --- the correction formed where it is used (pool factors 2, 4, 8) -----------------------
// For a compile-time p the node p*Z + a lies at u = Z + (2a - p + 1) / (2p) with -p < 2a-p+1 <
// 3p: its two voxels are the rows (Z-1, Z) for negative, (Z, Z+1) for other a, and its weight
// depends on a alone (a power-of-two quotient, exact), so a lane interpolates along x once per
// coarse row and then along y and z from registers, in apply_kernel's order: e is never stored.
template <int P>
struct Frac {
  static constexpr int num(int a) { return 2 * a - P + 1; }             // 2p * (u - Z)
  static constexpr int row(int a) { return num(a) < 0 ? 0 : 1; }        // of Z-1, Z, Z+1
  static constexpr float w(int a) {
    return static_cast<float>(num(a) < 0 ? num(a) + 2 * P : num(a)) / static_cast<float>(2 * P);
  }
};

__device__ __forceinline__ int clampi(int v, int hi) { return v < 0 ? 0 : (v > hi ? hi : v); }

// x-interpolated values of the coarse rows (Z-1..Z+1) x (Y-1..Y+1) at fine k.
__device__ __forceinline__ void x_rows(const float* __restrict__ out, int R, int p, int Z, int Y,
                                       int k, float (&c)[3][3]) {
  int x0, x1;
  float wx;
  interp_axis(k, p, R, x0, x1, wx);
#pragma unroll
  for (int z = 0; z < 3; ++z)
#pragma unroll
    for (int y = 0; y < 3; ++y) {
      const float* row = out + (static_cast<int64_t>(clampi(Z - 1 + z, R - 1)) * R +
                                clampi(Y - 1 + y, R - 1)) * R;
      c[z][y] = row[x0] * (1.0f - wx) + row[x1] * wx;
    }
}

template <int P>
__device__ __forceinline__ float yz_value(const float (&c)[3][3], int a, int b, float so) {
  const int z = Frac<P>::row(a), y = Frac<P>::row(b);
  const float wz = Frac<P>::w(a), wy = Frac<P>::w(b);
  const float c0 = c[z][y] * (1.0f - wy) + c[z][y + 1] * wy;
  const float c1 = c[z + 1][y] * (1.0f - wy) + c[z + 1][y + 1] * wy;
  return so * (c0 * (1.0f - wz) + c1 * wz);
}

// phi += e; a wave takes the nodes b = wave, wave + 4, ... of its slab.
template <int P>
__global__ void __launch_bounds__(256) update_net_kernel(const float* __restrict__ out, int R,
                                                         int n, const float* __restrict__ scales,
                                                         float* __restrict__ phi) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const Slab q = slab_of(pm::xcd_block(), R, (n + kSeg - 1) / kSeg);
  const int k = q.seg * kSeg + lane;
  if (k >= n || wave >= P) return;  // no barriers below
  constexpr int kB = (P + 3) / 4;  // b values per wave
  const bool kin = k >= 1 && k <= n - 2;
  float* const base = phi + (static_cast<int64_t>(P * q.Z) * n + P * q.Y) * n + k;
  float old[kB][P];
#pragma unroll
  for (int m = 0; m < kB; ++m)
#pragma unroll
    for (int a = 0; a < P; ++a)
      old[m][a] = base[(static_cast<int64_t>(a) * n + wave + 4 * m) * n];
  float c[3][3];
  x_rows(out, R, P, q.Z, q.Y, k, c);
  const float so = scales[3];
  __builtin_amdgcn_sched_barrier(0);  // all loads leave before any arithmetic
#pragma unroll
  for (int b = 0; b < P; ++b) {
    if ((b & 3) != wave) continue;
    const int j = P * q.Y + b;
#pragma unroll
    for (int a = 0; a < P; ++a) {
      const int i = P * q.Z + a;
      const float e = yz_value<P>(c, a, b, so);
      const bool in = i >= 1 && i <= n - 2 && j >= 1 && j <= n - 2 && kin;
      base[(static_cast<int64_t>(a) * n + b) * n] = old[b >> 2][a] + (in ? e : 0.0f);
    }
  }
}

// guard_kernel with e formed in LDS on the slab and its ring of one node instead of read: the
// same residuals, means and sums bit for bit (a wave takes the same nodes in the same order).
// Bound by instructions (the stencil in float64, the interpolation on the ring): 102 us at
// 256^3, where apply_kernel and guard_kernel took 62 + 63, the update 35 (36 now, with e formed
// again) and the split copy of the new residual, written split here, 46.
template <int P>
__global__ void __launch_bounds__(256) guard_net_kernel(const float* __restrict__ r32,
                                                        const float* __restrict__ out, int n,
                                                        int R, double inv_h2,
                                                        const float* __restrict__ scales,
                                                        float* __restrict__ rnew, int hn,
                                                        double* __restrict__ partials) {
  constexpr int W = P + 2, kRow = kSeg + 2;
  constexpr int kPer = (P * P + 3) / 4;  // nodes per lane
  __shared__ float s[4][kSeg][2];
  __shared__ double s_red[4 * 3];
  __shared__ float s_e[W * W * kRow];
  double v[3] = {0.0, 0.0, 0.0};
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nseg = (n + kSeg - 1) / kSeg;
  const int64_t slabs = static_cast<int64_t>(R) * R * nseg;
  const float inv = 1.0f / static_cast<float>(P * P * P);
  const float so = scales[3];
  for (int64_t sl = blockIdx.x; sl < slabs; sl += gridDim.x) {
    const Slab q = slab_of(sl, R, nseg);
    const int k = q.seg * kSeg + lane;
    float rv[kPer];
#pragma unroll
    for (int m = 0; m < kPer; ++m) {
      const int ab = wave + 4 * m, i = P * q.Z + ab / P, j = P * q.Y + ab % P;
      rv[m] = (k < n && ab < P * P) ? r32[(static_cast<int64_t>(i) * n + j) * n + k] : 0.0f;
    }
    auto inside = [&](int i, int j, int kk) {
      return i >= 1 && i <= n - 2 && j >= 1 && j <= n - 2 && kk >= 1 && kk <= n - 2;
    };
    {
      float c[3][3];
      x_rows(out, R, P, q.Z, q.Y, k < n ? k : n - 1, c);
#pragma unroll
      for (int bj = 0; bj < W; ++bj) {
        if ((bj & 3) != wave) continue;
#pragma unroll
        for (int ai = 0; ai < W; ++ai)
          s_e[(ai * W + bj) * kRow + lane + 1] =
              inside(P * q.Z + ai - 1, P * q.Y + bj - 1, k) ? yz_value<P>(c, ai - 1, bj - 1, so)
                                                            : 0.0f;
      }
    }
    // the ring's two ends along k
    for (int t = threadIdx.x; t < 2 * W * W; t += blockDim.x) {
      const int ab = t >> 1, ai = ab / W, bj = ab - ai * W;
      const int kk = (t & 1) ? q.seg * kSeg + kSeg : q.seg * kSeg - 1;
      const int i = P * q.Z + ai - 1, j = P * q.Y + bj - 1;
      s_e[ab * kRow + ((t & 1) ? kSeg + 1 : 0)] =
          inside(i, j, kk) ? so * trilinear(out, R, P, i, j, kk) : 0.0f;
    }
    __syncthreads();
    float t[2] = {0.0f, 0.0f};
#pragma unroll
    for (int m = 0; m < kPer; ++m) {
      const int ab = wave + 4 * m, i = P * q.Z + ab / P, j = P * q.Y + ab % P;
      if (k < n && ab < P * P) {
        const float* e = s_e + ((ab / P + 1) * W + ab % P + 1) * kRow + lane + 1;
        double ra = 0.0, rb = 0.0;
        if (inside(i, j, k)) {
          const double sum = static_cast<double>(e[W * kRow]) + static_cast<double>(e[-W * kRow]) +
                             static_cast<double>(e[kRow]) + static_cast<double>(e[-kRow]) +
                             static_cast<double>(e[1]) + static_cast<double>(e[-1]);
          rb = static_cast<double>(rv[m]);
          ra = rb - (sum - 6.0 * static_cast<double>(e[0])) * inv_h2;
        }
        rnew[place(i, j, k, n, hn)] = static_cast<float>(ra);
        v[2] = v[2] + ra * ra;
        t[0] += static_cast<float>(rb);
        t[1] += static_cast<float>(ra);
      }
    }
    slab_reduce<2>(t, P, s);  // (its barriers also end the reads of s_e)
    if (wave == 0 && k < n && lane % P == 0) {
      const double mb = static_cast<double>(t[0] * inv), ma = static_cast<double>(t[1] * inv);
      v[0] = v[0] + mb * mb;
      v[1] = v[1] + ma * ma;
    }
  }
  pm::block_sum<3>(v, s_red);
  if (threadIdx.x == 0)
    for (int c = 0; c < 3; ++c) partials[blockIdx.x * pm::kRedMaxQ + c] = v[c];
}

// tgt[V] = mean over V's fine nodes of (phi - cand), times scales[4].
__global__ void __launch_bounds__(256) target_kernel(const float* __restrict__ phi,
                                                     const float* __restrict__ cand, int n, int p,
                                                     int R, const float* __restrict__ scales,
                                                     float* __restrict__ tgt) {
  const int64_t V = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t nv = static_cast<int64_t>(R) * R * R;
  if (V >= nv) return;
  const int X = static_cast<int>(V % R), Y = static_cast<int>((V / R) % R),
            Z = static_cast<int>(V / (static_cast<int64_t>(R) * R));
  float s = 0.0f;
  for (int a = 0; a < p; ++a)
    for (int b = 0; b < p; ++b) {
      const int64_t base = (static_cast<int64_t>(p * Z + a) * n + (p * Y + b)) * n + p * X;
      for (int c = 0; c < p; ++c) s += phi[base + c] - cand[base + c];
    }
  tgt[V] = s / static_cast<float>(p * p * p) * scales[4];
}

}  // namespace

namespace pm {
namespace warm {

pm_status extrapolate(float* phi, float* hist, float* cand, int n, hipStream_t s) {
  const int64_t total = static_cast<int64_t>(n) * n * n;
  PM_TIMED("warm.extrapolate", (cand ? 20.0 : 16.0) * static_cast<double>(total), s);
  const uintptr_t bits = reinterpret_cast<uintptr_t>(phi) | reinterpret_cast<uintptr_t>(hist) |
                         reinterpret_cast<uintptr_t>(cand);
  if (n % 4 == 0 && (bits & 15u) == 0)
    extrap4_kernel<<<pm::blocks_for(total / 4), pm::kBlock, 0, s>>>(phi, hist, cand, n);
  else
    extrap_kernel<<<pm::blocks_for(total), pm::kBlock, 0, s>>>(phi, hist, cand, n);
  PM_CHECK_LAUNCH("extrap_kernel");
  return PM_OK;
}

pm_status make_input(const float* r32, const float* phi, const float* hist, const float* rho,
                     float factor, int n, int p, double h, float* pooled, uint16_t* input, double* partials,
                     double* red, float* scales, hipStream_t s) {
  PM_REQUIRE(p >= 1 && p <= kSeg && kSeg % p == 0 && n % p == 0,
             "warm start: the pool factor must divide 64 and the grid size");
  const int R = n / p;
  const int64_t nv = static_cast<int64_t>(R) * R * R;
  const int nseg = (n + kSeg - 1) / kSeg;
  const int64_t slabs = static_cast<int64_t>(R) * R * nseg;
  const unsigned blocks = static_cast<unsigned>(std::min<int64_t>(slabs, pm::kRedBlocks));
  {
    PM_TIMED("warm.input", 16.0 * static_cast<double>(n) * n * n, s);
    pool_input_kernel<<<blocks, pm::kBlock, 0, s>>>(r32, phi, hist, rho, factor, n, p, R, pooled,
                                                      partials);
    PM_CHECK_LAUNCH("pool_input_kernel");
    pm::fold_partials_kernel<3><<<1, pm::kBlock, 0, s>>>(partials, static_cast<int>(blocks), red);
    PM_CHECK_LAUNCH("fold_partials_kernel<3>");
    scales_kernel<<<1, 64, 0, s>>>(red, nv, (p * h) * (p * h), scales);
    PM_CHECK_LAUNCH("scales_kernel");
    normalize_kernel<<<pm::blocks_for(nv), pm::kBlock, 0, s>>>(pooled, nv, scales, input);
    PM_CHECK_LAUNCH("normalize_kernel");
  }
  return PM_OK;
}

bool fused(int p) { return p == 2 || p == 4 || p == 8; }

pm_status guard(const float* r32, const float* out, int n, int p, double h, const float* scales,
                float* e, float* rnew, int hn, double* partials, double* red, hipStream_t s) {
  const int R = n / p;
  const int64_t slabs = static_cast<int64_t>(R) * R * ((n + kSeg - 1) / kSeg);
  const unsigned b = static_cast<unsigned>(std::min<int64_t>(slabs, pm::kRedBlocks));
  const double nodes = static_cast<double>(n) * n * n, inv_h2 = 1.0 / (h * h);
  if (fused(p)) {
    PM_TIMED("warm.guard", 8.0 * nodes, s);
#define PM_GUARD(P)                                                                            \
  guard_net_kernel<P><<<b, pm::kBlock, 0, s>>>(r32, out, n, R, inv_h2, scales, rnew, hn, partials)
    if (p == 2)
      PM_GUARD(2);
    else if (p == 4)
      PM_GUARD(4);
    else
      PM_GUARD(8);
#undef PM_GUARD
    PM_CHECK_LAUNCH("guard_net_kernel");
  } else {
    PM_TIMED("warm.guard", 16.0 * nodes, s);
    apply_kernel<<<static_cast<unsigned>(slabs), pm::kBlock, 0, s>>>(out, R, p, n, scales, e);
    PM_CHECK_LAUNCH("apply_kernel");
    guard_kernel<<<b, pm::kBlock, 0, s>>>(r32, e, n, p, R, inv_h2, rnew, hn, partials);
    PM_CHECK_LAUNCH("guard_kernel");
  }
  pm::fold_partials_kernel<3><<<1, pm::kBlock, 0, s>>>(partials, static_cast<int>(b), red);
  PM_CHECK_LAUNCH("fold_partials_kernel<3>");
  return PM_OK;
}

pm_status correct(float* phi, const float* out, int n, int p, const float* scales, const float* e,
                  hipStream_t s) {
  const int R = n / p;
  const int64_t slabs = static_cast<int64_t>(R) * R * ((n + kSeg - 1) / kSeg);
  const int64_t nodes = static_cast<int64_t>(n) * n * n;
  const unsigned b = static_cast<unsigned>(slabs);
  PM_TIMED("warm.correct", (fused(p) ? 8.0 : 12.0) * static_cast<double>(nodes), s);
  if (p == 2)
    update_net_kernel<2><<<b, pm::kBlock, 0, s>>>(out, R, n, scales, phi);
  else if (p == 4)
    update_net_kernel<4><<<b, pm::kBlock, 0, s>>>(out, R, n, scales, phi);
  else if (p == 8)
    update_net_kernel<8><<<b, pm::kBlock, 0, s>>>(out, R, n, scales, phi);
  else
    add_kernel<<<pm::blocks_for(nodes), pm::kBlock, 0, s>>>(phi, e, nodes);
  PM_CHECK_LAUNCH("update_net_kernel");
  return PM_OK;
}

pm_status target(const float* phi, const float* cand, int n, int p, const float* scales, float* tgt,
                 hipStream_t s) {
  const int R = n / p;
  const int64_t nv = static_cast<int64_t>(R) * R * R;
  PM_TIMED("warm.target", 8.0 * static_cast<double>(n) * n * n, s);
  target_kernel<<<pm::blocks_for(nv), pm::kBlock, 0, s>>>(phi, cand, n, p, R, scales, tgt);
  PM_CHECK_LAUNCH("target_kernel");
  return PM_OK;
}

}  // namespace warm
}  // namespace pm
