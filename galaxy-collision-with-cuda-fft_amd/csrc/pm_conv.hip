// BF16 3x3x3 convolutions on the gfx950 matrix cores, for the learned multigrid warm start.
//
// Tensors are channels-last: element (voxel v, channel c) of an r^3 tensor with C channels
// sits at v*C + c, v = (z*r + y)*r + x (x fastest, the grid's k axis). BF16 values travel as
// their 16-bit patterns (uint16_t). Every convolution is "same" (zero padding 1, stride 1)
// and cross-correlates like torch.nn.functional.conv3d:
//     y[v][co] = bias[co] + sum_{ci, tap} w[co][ci][tap] * x[v + off(tap)][ci],
//     tap = (dz+1)*9 + (dy+1)*3 + (dx+1), off(tap) = (dz, dy, dx).
// The input may be the concatenation of two tensors: xa (ca channels) then xb (cb channels);
// with up_a set, xa lives at resolution r/2 and is read nearest-neighbour upsampled, which
// is the decoder's "upsample, concatenate the skip, convolve" fused into the operand loads.
//
// Forward is an implicit GEMM: rows = output voxels, columns = output channels, reduction
// k = tap*Cin + ci over packed weights w_p[co][k] (bf16, rows padded to 16, k to 32). Each
// wave computes 64 voxels x Cout with v_mfma_f32_16x16x32_bf16 (float32 accumulation).
// Backward-data is the forward kernel applied to dZ with the weights flipped in space and
// transposed in channels. Backward-weight reduces over voxels: dW[co][k] = sum_v dZ[v][co] *
// im2col(x)[v][k]; both operands are staged transposed through LDS so that the 32-voxel
// reduction chunk is contiguous per lane, partial sums per voxel split are written and
// folded in a fixed order (deterministic).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "pm_common.h"
#include "pm_conv.h"
#include "pm_timing.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

using pm::conv::bf2f;
using pm::conv::f2bf;

__device__ __forceinline__ f32x4_t mfma_bf16(u32x4_t a, u32x4_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                  __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

__device__ __forceinline__ u32x4_t load16(const uint16_t* p) {
  return *reinterpret_cast<const u32x4_t*>(p);
}

struct ConvFwdArgs {
  const uint16_t* xa;
  const uint16_t* xb;
  int ca, cb, cin, r, ra, up;
  const uint16_t* w;  // packed operands (pack_weights_kernel)
  int kpad, kreal, rows;
  int kc_per;         // 32-wide reduction chunks per split (blockIdx.z)
  float* partial;     // split-K: raw sums [split][r^3][rows] (epilogue in a second kernel)
  const float* bias;
  int cout, cout_st, act;
  float slope;
  uint16_t* y;   // [r^3][cout_st] or null
  float* y32;    // [r^3][cout] or null
};

// Source element (voxel (z, y, x) of the concatenated input, channels ci..ci+7) or null
// when the voxel lies outside the r^3 box (zero padding).
__device__ __forceinline__ const uint16_t* conv_src(const uint16_t* xa, const uint16_t* xb, int ca,
                                                    int cb, int r, int ra, int up, int z, int y,
                                                    int x, int ci) {
  if (static_cast<unsigned>(z) >= static_cast<unsigned>(r) ||
      static_cast<unsigned>(y) >= static_cast<unsigned>(r) ||
      static_cast<unsigned>(x) >= static_cast<unsigned>(r))
    return nullptr;
  if (ci < ca) {
    const int idx = up ? ((z >> 1) * ra + (y >> 1)) * ra + (x >> 1) : (z * r + y) * r + x;
    return xa + static_cast<int64_t>(idx) * ca + ci;
  }
  return xb + static_cast<int64_t>((z * r + y) * r + x) * cb + (ci - ca);
}

// One wave: 64 output voxels (4 MFMA row blocks) x output channels co0 .. co0 + 16*NB - 1,
// co0 = blockIdx.y * 16 * NB (column blocks at or beyond the packed weight rows are
// skipped), over the reduction chunks of split blockIdx.z.
template <int NB>
__global__ void __launch_bounds__(256) conv_fwd_kernel(ConvFwdArgs a) {
  const int co0 = static_cast<int>(blockIdx.y) * 16 * NB;
  const int kbeg = static_cast<int>(blockIdx.z) * a.kc_per * 32;
  const int kend = min(a.kpad, kbeg + a.kc_per * 32);
  const int lane = threadIdx.x & 63;
  const int row = lane & 15, grp = lane >> 4;
  const int r = a.r;
  const int nvox = r * r * r;
  const int vbase = (static_cast<int>(pm::xcd_block()) * 4 + static_cast<int>(threadIdx.x >> 6)) * 64;
  if (vbase >= nvox) return;  // whole wave idle (no barriers in this kernel)

  int vz[4], vy[4], vx[4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) {
    const int v = vbase + 16 * mb + row;
    if (v < nvox) {
      vx[mb] = v % r;
      vy[mb] = (v / r) % r;
      vz[mb] = v / (r * r);
    } else {
      vz[mb] = -4;  // every neighbour of this row falls outside the box
      vy[mb] = vx[mb] = 0;
    }
  }
  f32x4_t acc[4][NB];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // this lane's k = kc + 8*grp as (tap, ci); advanced by 32 per chunk
  int tap = (kbeg + 8 * grp) / a.cin;
  int ci = kbeg + 8 * grp - tap * a.cin;
  const uint16_t* wrow[NB];
  bool wvalid[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    wvalid[nb] = co0 + 16 * nb < a.rows;
    wrow[nb] = a.w + static_cast<int64_t>(wvalid[nb] ? co0 + 16 * nb : 0) * a.kpad + 8 * lane;
  }

  // G consecutive 32-wide chunks per round: every operand load of the round is issued
  // before its first MFMA (a chunk's few MFMAs cannot hide a load's latency on their own),
  // and the chunks are accumulated in order, as one chunk per round would
  constexpr int G = NB <= 2 ? 2 : 1;
  for (int kc = kbeg; kc < kend; kc += 32 * G) {
    u32x4_t av[G][4];
    u32x4_t bv[G][NB];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int kcg = kc + 32 * g;
      const bool live = kcg < kend;
      const bool kin = live && kcg + 8 * grp < a.kreal;
      const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) {
        const uint16_t* p = kin ? conv_src(a.xa, a.xb, a.ca, a.cb, r, a.ra, a.up, vz[mb] + dz,
                                           vy[mb] + dy, vx[mb] + dx, ci)
                                : nullptr;
        av[g][mb] = p ? load16(p) : u32x4_t{0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        bv[g][nb] = (live && wvalid[nb]) ? load16(wrow[nb] + 16 * kcg) : u32x4_t{0u, 0u, 0u, 0u};
      ci += 32;
      while (ci >= a.cin) {
        ci -= a.cin;
        ++tap;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (kc + 32 * g >= kend) break;  // uniform
#pragma unroll
      for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          acc[mb][nb] = mfma_bf16(av[g][mb], bv[g][nb], acc[mb][nb]);
    }
  }

  // D layout: lane holds rows 4*grp + i (voxels), column `row` (output channel)
  if (a.partial) {
    float* out = a.partial + static_cast<int64_t>(blockIdx.z) * nvox * a.rows;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int co = co0 + 16 * nb + row;
      if (co >= a.rows) continue;
#pragma unroll
      for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int v = vbase + 16 * mb + 4 * grp + i;
          if (v < nvox) out[static_cast<int64_t>(v) * a.rows + co] = acc[mb][nb][i];
        }
    }
    return;
  }
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int co = co0 + 16 * nb + row;
    if (co >= a.cout_st) continue;
    const bool real = co < a.cout;
    const float b = (real && a.bias) ? a.bias[co] : 0.0f;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int v = vbase + 16 * mb + 4 * grp + i;
        if (v >= nvox) continue;
        float val = 0.0f;
        if (real) {
          val = acc[mb][nb][i] + b;
          if (a.act && !(val > 0.0f)) val = val * a.slope;
        }
        if (a.y) a.y[static_cast<int64_t>(v) * a.cout_st + co] = f2bf(val);
        if (a.y32 && real) a.y32[static_cast<int64_t>(v) * a.cout + co] = val;
      }
    }
  }
}

// The forward convolution from an LDS tile: a workgroup stages the input of a 2 x 8 x 8 block of
// output voxels with its halo once (4 x 10 x 10 voxels, all CIN input channels) and its waves
// read every tap's operand from there, where conv_fwd_kernel loads each activation 27 times
// through the caches and decodes its address each time (us, both with 256 threads: 16 -> 16 at
// 64^3 24 there, 12 here; 48 -> 16 at 64^3 54, 27; 96 -> 32 at 32^3 37 + 5 for its split sums, 17;
// 128 -> 128 at 8^3 10 + 9, 19; 192 -> 64 at 16^3 25 + 5, 28). Bound: LDS operand reads and the
// staging's latency. Wave w computes voxels 32 w .. 32 w + 31
// x 16 * NB output channels over the reduction in packed order, as one split of conv_fwd_kernel
// does. The reduction is unrolled: a chunk of 32 is one weight load, two LDS reads and 2 * NB
// MFMAs, its addresses constant offsets (computed per chunk, in vector or scalar registers, they
// took several times as long as the MFMAs). A voxel's channels are padded by 16 bytes so that
// the 16 rows of an operand read fall into different banks.
constexpr int kHaloY = 10, kHaloZ = 100;   // strides of the staged 4 x 10 x 10 voxels
constexpr int kHaloVox = 400;

constexpr int tap_offset(int tap) {  // staged voxels from the block's first; taps past 26 read one
  return tap > 26 ? 0 : (tap / 9) * kHaloZ + (tap / 3 % 3) * kHaloY + tap % 3;
}

struct ConvTileArgs {
  ConvFwdArgs c;
  pm::FastDiv dt;         // 8 x 8 blocks of a plane per axis
};

// S > 1: the channels are staged in S slices, one after the other (less LDS, so that another
// workgroup computes while this one stages).
template <int CIN, int NB, int S>
__global__ void __launch_bounds__(256) conv_tile_kernel(ConvTileArgs t) {
  extern __shared__ __align__(16) unsigned char lds[];
  constexpr int CS = CIN / S;  // channels staged at once
  static_assert(S == 1 || CS % 32 == 0, "a slice is whole chunks of every tap");
  constexpr int kPitch = 2 * CS + 16;
  constexpr int kReal = 27 * CS, kChunks = (kReal + 31) / 32;  // of a slice
  const ConvFwdArgs& a = t.c;
  const int r = a.r;
  const uint32_t blk = static_cast<uint32_t>(pm::xcd_block());
  const uint32_t q0 = pm::fast_div(blk, t.dt), q1 = pm::fast_div(q0, t.dt);
  const int x0 = static_cast<int>(blk - q0 * t.dt.d) * 8;
  const int y0 = static_cast<int>(q0 - q1 * t.dt.d) * 8;
  const int z0 = static_cast<int>(q1) * 2;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = lane & 15, grp = lane >> 4;
  const int co0 = static_cast<int>(blockIdx.y) * 16 * NB;
  // weights of the first chunks leave before the staging
  constexpr int kAhead = NB == 1 ? 8 : 4;
  const uint16_t* wrow[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)  // a column block past the packed rows repeats the last one
    wrow[nb] = a.w + static_cast<int64_t>(min(co0 + 16 * nb, a.rows - 16)) * a.kpad + 8 * lane;
  u32x4_t bv[kAhead][NB];
  // weights of chunk c of slice s: all of a tap's channels are consecutive chunks
  auto weights = [&](int s, int c, u32x4_t (&dst)[NB]) {
    const int at = S == 1 ? c : c / (CS / 32) * (CIN / 32) + s * (CS / 32) + c % (CS / 32);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) dst[nb] = load16(wrow[nb] + 512 * at);
  };
  const unsigned char* base[2];
  const bool second = grp >= 2;
#pragma unroll
  for (int mb = 0; mb < 2; ++mb) {
    const int m = 32 * wave + 16 * mb + row;
    base[mb] = lds + ((m >> 6) * kHaloZ + ((m >> 3) & 7) * kHaloY + (m & 7)) * kPitch;
  }
  f32x4_t acc[2][NB];
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int slice = 0; slice < S; ++slice) {
#pragma unroll
    for (int c = 0; c < kAhead && c < kChunks; ++c) weights(slice, c, bv[c]);
    if (slice > 0) __syncthreads();  // the previous slice has been read
    {
      // thread -> one (x, 8 channels) of a staged row and every kRows-th of the 40 rows: source
      // tensor, channel and x are found once
      constexpr int kItems = kHaloY * (CS / 8), kRows = 256 / kItems;
      constexpr int kRounds = (40 + kRows - 1) / kRows;
      constexpr int kBatch = kRounds < 10 ? kRounds : 10;  // loads in flight per thread
      const int rr = static_cast<int>(threadIdx.x) / kItems;
      const int item = static_cast<int>(threadIdx.x) - rr * kItems;
      const int hx = item / (CS / 8), c8 = 8 * (item - hx * (CS / 8)), g8 = slice * CS + c8;
      const bool from_a = g8 < a.ca;
      const int sh = from_a ? a.up : 0, rs = from_a ? a.ra : r, cs = from_a ? a.ca : a.cb;
      const int x = x0 + hx - 1;
      const uint16_t* src = (from_a ? a.xa + g8 : a.xb + (g8 - a.ca)) + (x >> sh) * cs;
      const bool x_in = rr < kRows && x >= 0 && x < r;
      unsigned char* dst = lds + hx * kPitch + 2 * c8;
#pragma unroll
      for (int u0 = 0; u0 < kRounds; u0 += kBatch) {
        u32x4_t v[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          const int rowi = rr + (u0 + u) * kRows;
          const int hz = (rowi * 205) >> 11, hy = rowi - 10 * hz;  // rowi / 10 for rowi < 80
          const int z = z0 + hz - 1, y = y0 + hy - 1;
          const bool in = u0 + u < kRounds && rowi < 40 && x_in && z >= 0 && z < r && y >= 0 && y < r;
          const int vrow = __mul24(__mul24(z >> sh, rs) + (y >> sh), rs);
          v[u] = in ? load16(src + static_cast<int64_t>(vrow) * cs) : u32x4_t{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          const int rowi = rr + (u0 + u) * kRows;
          if (u0 + u < kRounds && rowi < 40 && rr < kRows)
            *reinterpret_cast<u32x4_t*>(dst + rowi * (kHaloY * kPitch)) = v[u];
        }
      }
    }
    __syncthreads();
    // operand address of row block mb: base + the chunk's constant; where the chunk's two halves
    // (16 channels each) lie in different taps, the lanes of the second half add the taps'
    // distance: one voxel along x, or to the next row or plane
    constexpr int kReads = 3;  // chunks whose LDS reads are under way
    u32x4_t av[kReads][2];
    auto operand = [&](int c, u32x4_t (&dst)[2]) {
      // byte offsets of the chunk's four operand groups (8 channels each)
      int off[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int k = 32 * c + 8 * g;
        off[g] = tap_offset(k / CS) * kPitch + 2 * (k % CS);
      }
      int lane_off;
      if (CS % 16 == 0) {
        const int jump = off[2] - off[0] - 32;  // 0 where the chunk lies in one tap
        lane_off = 16 * grp + (second ? jump : 0) + off[0];
      } else {
        lane_off = grp == 0 ? off[0] : grp == 1 ? off[1] : grp == 2 ? off[2] : off[3];
      }
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) dst[mb] = *reinterpret_cast<const u32x4_t*>(base[mb] + lane_off);
      if (32 * (c + 1) > kReal) {  // the last chunk's padding: weights there are zero, so must x be
        const bool in = 32 * c + 8 * grp < kReal;
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) dst[mb] = in ? dst[mb] : u32x4_t{0u, 0u, 0u, 0u};
      }
    };
#pragma unroll
    for (int c = 0; c < kReads && c < kChunks; ++c) operand(c, av[c]);
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          acc[mb][nb] = mfma_bf16(av[c % kReads][mb], bv[c % kAhead][nb], acc[mb][nb]);
      if (c + kReads < kChunks) operand(c + kReads, av[c % kReads]);
      if (c + kAhead < kChunks) weights(slice, c + kAhead, bv[c % kAhead]);
    }
  }
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int co = co0 + 16 * nb + row;
    if (co >= a.cout_st) continue;
    const bool real = co < a.cout;
    const float b = (real && a.bias) ? a.bias[co] : 0.0f;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = 32 * wave + 16 * mb + 4 * grp + i;
        const int z = z0 + (m >> 6), y = y0 + ((m >> 3) & 7), x = x0 + (m & 7);
        if (z >= r || y >= r || x >= r) continue;
        const int v = (z * r + y) * r + x;
        float val = 0.0f;
        if (real) {
          val = acc[mb][nb][i] + b;
          if (a.act && !(val > 0.0f)) val = val * a.slope;
        }
        if (a.y) a.y[static_cast<int64_t>(v) * a.cout_st + co] = f2bf(val);
        if (a.y32 && real) a.y32[static_cast<int64_t>(v) * a.cout + co] = val;
      }
    }
  }
}

// Split-K epilogue: y = act(bias + sum over splits in order), one thread per output value.
__global__ void __launch_bounds__(256) conv_epilogue_kernel(const float* __restrict__ partial,
                                                            int splits, int nvox, int rows,
                                                            const float* __restrict__ bias,
                                                            int cout, int cout_st, int act,
                                                            float slope, uint16_t* y, float* y32) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= static_cast<int64_t>(nvox) * cout_st) return;
  const int co = static_cast<int>(idx % cout_st);
  const int v = static_cast<int>(idx / cout_st);
  float val = 0.0f;
  if (co < cout) {
    float sum = 0.0f;
    for (int z = 0; z < splits; ++z)
      sum += partial[(static_cast<int64_t>(z) * nvox + v) * rows + co];
    val = sum + (bias ? bias[co] : 0.0f);
    if (act && !(val > 0.0f)) val = val * slope;
  }
  if (y) y[idx] = f2bf(val);
  if (y32 && co < cout) y32[static_cast<int64_t>(v) * cout + co] = val;
}

struct ConvWgradArgs {
  const uint16_t* xa;
  const uint16_t* xb;
  int ca, cb, cin, r, ra, up;
  const uint16_t* dz;  // [r^3][dz_c]
  int dz_c, kreal, nvox, chunks_per_split;
  float* partial;      // [splits][16*NR][kcols]
  int kcols;
  float* partial_b;    // [splits][16*NR] channel sums of dz, or null
};

// grid (kcols/64, splits): one workgroup = 64 reduction columns x all output channels over
// one voxel range; wave w owns columns 16w..16w+15. The first column group's wave 0 also
// multiplies dz with ones: the bias gradient's sums ride on operands it has loaded anyway
// (a pass of their own took 31-118 us a layer at 64^3-16^3, as long as this kernel).
//
// A stage of V voxels is loaded a stage ahead into registers and transposed into LDS as pairs of
// voxels (one 32-bit write per two); both operands then come from LDS for V/32 products. Staging
// 32 voxels at a time with their loads waited for in place, and coordinates by division, took 60
// us a call over the layers of 16 channels at 64^3-8^3 (now 38), 22 at 32 channels (18), 16 at
// 64 (14). Above 64 rows the LDS tile and the few voxels of those layers want V = 64.
template <int NR, int V>
__global__ void __launch_bounds__(256) conv_wgrad_kernel(ConvWgradArgs a) {
  constexpr int kLd = V + 8;       // row stride: keeps 16-byte alignment
  constexpr int kXP = V / 64;      // voxel pairs of x per thread and stage
  constexpr int kDP = NR * V >= 256 ? NR * V / 256 : 1;  // pair loads of dz per thread, at most
  __shared__ __align__(16) uint16_t sdz[NR * 16][kLd];
  __shared__ __align__(16) uint16_t sx[64][kLd];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int row = lane & 15, grp = lane >> 4;
  const int k0 = blockIdx.x * 64;
  const int split = blockIdx.y;

  for (int p = tid; p < NR * 16 * kLd; p += 256) (&sdz[0][0])[p] = 0;  // rows >= dz_c stay 0

  const int cg = tid >> 5, vs = tid & 31;  // x staging: column group (8 columns), pair slot
  const int kq = k0 + 8 * cg;
  const bool kvalid = kq < a.kreal;
  int ci = 0, dz = 0, dy = 0, dx = 0;
  if (kvalid) {
    const int tap = kq / a.cin;
    ci = kq - tap * a.cin;
    dz = tap / 9 - 1;
    dy = (tap / 3) % 3 - 1;
    dx = tap % 3 - 1;
  }
  const int c8s = __builtin_ctz(static_cast<unsigned>(a.dz_c)) - 3;  // dz_c / 8 = 1 << c8s
  const bool pow2 = (a.r & (a.r - 1)) == 0;
  const int rs = __builtin_ctz(static_cast<unsigned>(a.r));
  f32x4_t acc[NR];
#pragma unroll
  for (int rb = 0; rb < NR; ++rb) acc[rb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const bool sums = a.partial_b && blockIdx.x == 0 && wave == 0;
  f32x4_t accb[NR];
#pragma unroll
  for (int rb = 0; rb < NR; ++rb) accb[rb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const u32x4_t ones = u32x4_t{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};

  const int vbeg = split * a.chunks_per_split * 32;
  const int vend = min(a.nvox, vbeg + a.chunks_per_split * 32);
  u32x4_t xr[kXP][2], dr[kDP][2];
  auto load_stage = [&](int vc) {
#pragma unroll
    for (int m = 0; m < kXP; ++m)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int v = vc + 64 * m + 2 * vs + h;
        xr[m][h] = u32x4_t{0u, 0u, 0u, 0u};
        if (kvalid && v < vend) {
          int x, y, z;
          if (pow2) {
            x = v & (a.r - 1);
            y = (v >> rs) & (a.r - 1);
            z = v >> (2 * rs);
          } else {
            x = v % a.r;
            y = (v / a.r) % a.r;
            z = v / (a.r * a.r);
          }
          const uint16_t* p =
              conv_src(a.xa, a.xb, a.ca, a.cb, a.r, a.ra, a.up, z + dz, y + dy, x + dx, ci);
          if (p) xr[m][h] = load16(p);
        }
      }
#pragma unroll
    for (int m = 0; m < kDP; ++m)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int p = tid + 256 * m, vp = p >> c8s, c8 = p & ((1 << c8s) - 1);
        const int v = vc + 2 * vp + h;
        dr[m][h] = u32x4_t{0u, 0u, 0u, 0u};
        if (vp < V / 2 && v < vend)
          dr[m][h] = load16(a.dz + static_cast<int64_t>(v) * a.dz_c + 8 * c8);
      }
  };
  // channels 8q..8q+7 of a voxel pair into 8 rows, one 32-bit write each
  auto put = [&](uint16_t* dst, const u32x4_t& lo, const u32x4_t& hi) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      *reinterpret_cast<uint32_t*>(dst + (2 * q) * kLd) = (lo[q] & 0xffffu) | (hi[q] << 16);
      *reinterpret_cast<uint32_t*>(dst + (2 * q + 1) * kLd) = (lo[q] >> 16) | (hi[q] & 0xffff0000u);
    }
  };
  if (vbeg < vend) load_stage(vbeg);
  for (int vc = vbeg; vc < vend; vc += V) {
    __syncthreads();  // the previous stage's MFMA reads are done (and the zero fill above)
#pragma unroll
    for (int m = 0; m < kDP; ++m) {
      const int p = tid + 256 * m, vp = p >> c8s, c8 = p & ((1 << c8s) - 1);
      if (vp < V / 2) put(&sdz[8 * c8][2 * vp], dr[m][0], dr[m][1]);
    }
#pragma unroll
    for (int m = 0; m < kXP; ++m) put(&sx[8 * cg][64 * m + 2 * vs], xr[m][0], xr[m][1]);
    __syncthreads();
    if (vc + V < vend) load_stage(vc + V);
#pragma unroll
    for (int q = 0; q < V / 32; ++q) {
      if (vc + 32 * q >= vend) break;
      const u32x4_t bq = *reinterpret_cast<const u32x4_t*>(&sx[16 * wave + row][32 * q + 8 * grp]);
#pragma unroll
      for (int rb = 0; rb < NR; ++rb) {
        const u32x4_t aq =
            *reinterpret_cast<const u32x4_t*>(&sdz[16 * rb + row][32 * q + 8 * grp]);
        acc[rb] = mfma_bf16(aq, bq, acc[rb]);
        if (sums) accb[rb] = mfma_bf16(aq, ones, accb[rb]);
      }
    }
  }
  if (sums && row == 0) {  // every column holds the same sums
#pragma unroll
    for (int rb = 0; rb < NR; ++rb)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        a.partial_b[split * (16 * NR) + 16 * rb + 4 * grp + i] = accb[rb][i];
  }
  const int kcol = k0 + 16 * wave + row;
#pragma unroll
  for (int rb = 0; rb < NR; ++rb)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int co = 16 * rb + 4 * grp + i;
      a.partial[(static_cast<int64_t>(split) * (16 * NR) + co) * a.kcols + kcol] = acc[rb][i];
    }
}

// dw[co][ci][tap] (torch layout) = (accumulate ? dw : 0) + the sum over splits, and db[co] the
// same of the channel sums. grid (kcols/64, cout + 1): 64 columns of one output channel (the
// last grid row: 64 channels of the bias); the kFoldWaves waves take every kFoldWaves-th split,
// a few loads in flight at once, and their sums are added in wave order (deterministic). One
// thread that walked all splits of an output kept a load at a time in flight: 80 us for the
// 283 splits that a 64^3 layer of 16 channels had, 157 us for 512.
constexpr int kFoldWaves = 16;
__global__ void __launch_bounds__(64 * kFoldWaves) wgrad_fold_kernel(
    const float* __restrict__ partial, const float* __restrict__ partial_b, int splits, int cout,
    int rows, int kcols, int cin, float* dw, float* db, int accumulate) {
  __shared__ float s[kFoldWaves][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = static_cast<int>(blockIdx.x) * 64 + lane;
  const bool bias = static_cast<int>(blockIdx.y) == cout;
  const int co = bias ? col : static_cast<int>(blockIdx.y);
  const bool live = bias ? db && col < cout : col < 27 * cin;
  const float* src = bias ? partial_b + col : partial + static_cast<int64_t>(co) * kcols + col;
  const int64_t stride = bias ? rows : static_cast<int64_t>(rows) * kcols;
  float sum = 0.0f;
  if (live) {
    constexpr int kAhead = 8;
    for (int sp = wave; sp < splits; sp += kFoldWaves * kAhead) {
      float v[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int at = sp + u * kFoldWaves;
        v[u] = at < splits ? src[at * stride] : 0.0f;
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u) sum += v[u];
    }
  }
  s[wave][lane] = sum;
  __syncthreads();
  if (wave != 0 || !live) return;
  float t = s[0][lane];
#pragma unroll
  for (int w = 1; w < kFoldWaves; ++w) t += s[w][lane];
  float* out = bias ? db + col
                    : dw + (static_cast<int64_t>(co) * cin + col % cin) * 27 + col / cin;
  *out = accumulate ? *out + t : t;
}

// Pack torch-layout float32 weights w[co][ci][27] into bf16 GEMM operands.
//   forward:   wp[co][tap*cin + ci]            rows co < rows_pad, k < kpad
//   transpose: wp[ci][tap'*cout_st + co] = w[co][ci][26 - tap']   (backward-data operand)
// stored by MFMA operand: 16 rows x 32 k are 512 consecutive values, lane 16 * (k / 8 % 4) +
// row % 16 holding 8 of them, so that a wave loads an operand as one contiguous kilobyte (as
// 16 rows of 64 bytes it kept the cache port busy for longer than the MFMAs took).
__global__ void __launch_bounds__(256) pack_weights_kernel(const float* __restrict__ w, int cout,
                                                           int cin, int transpose, int cin_eff,
                                                           int rows_pad, int kpad,
                                                           uint16_t* __restrict__ wp) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= static_cast<int64_t>(rows_pad) * kpad) return;
  const int lane = static_cast<int>(idx >> 3) & 63, chunks = kpad >> 5;
  const int block = static_cast<int>(idx >> 9);
  const int rrow = block / chunks * 16 + (lane & 15);
  const int k = block % chunks * 32 + (lane >> 4) * 8 + static_cast<int>(idx & 7);
  float v = 0.0f;
  if (k < 27 * cin_eff) {
    const int tap = k / cin_eff, c = k - tap * cin_eff;
    if (!transpose) {
      // rrow = co, c = ci
      if (rrow < cout && c < cin) v = w[(static_cast<int64_t>(rrow) * cin + c) * 27 + tap];
    } else {
      // rrow = ci, c = co (cin_eff = cout_st)
      if (rrow < cin && c < cout) v = w[(static_cast<int64_t>(c) * cin + rrow) * 27 + (26 - tap)];
    }
  }
  wp[idx] = f2bf(v);
}

// 2x2x2 average pooling, bf16 -> bf16 (float32 sum in a fixed order), C % 8 == 0.
__global__ void __launch_bounds__(256) pool2_kernel(const uint16_t* __restrict__ x, int r, int c,
                                                    uint16_t* __restrict__ y) {
  const int rc = r >> 1;
  const int groups = c >> 3;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= static_cast<int64_t>(rc) * rc * rc * groups) return;
  const int g = static_cast<int>(idx % groups);
  const int vc = static_cast<int>(idx / groups);
  const int X = vc % rc, Y = (vc / rc) % rc, Z = vc / (rc * rc);
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int child = 0; child < 8; ++child) {
    const int z = 2 * Z + (child >> 2), yy = 2 * Y + ((child >> 1) & 1), xx = 2 * X + (child & 1);
    const u32x4_t v = load16(x + static_cast<int64_t>((z * r + yy) * r + xx) * c + 8 * g);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      s[2 * q] += bf2f(static_cast<uint16_t>(v[q] & 0xffffu));
      s[2 * q + 1] += bf2f(static_cast<uint16_t>(v[q] >> 16));
    }
  }
  u32x4_t o;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    o[q] = static_cast<uint32_t>(f2bf(s[2 * q] * 0.125f)) |
           (static_cast<uint32_t>(f2bf(s[2 * q + 1] * 0.125f)) << 16);
  *reinterpret_cast<u32x4_t*>(y + static_cast<int64_t>(vc) * c + 8 * g) = o;
}

// dz[v][c] = bf16((g1[v][c] + g2[parent(v)][c] / 8) * act'(y[v][c])) for c < gc, 0 for the
// pad channels c in [gc, dz_c). g1 has stride g1_stride and may be null; g2 (the gradient
// of a following 2x2x2 average pool, at resolution r/2 with gc channels) may be null;
// y null means no activation (derivative 1).
__global__ void __launch_bounds__(256) act_bwd_kernel(const float* __restrict__ g1,
                                                      int g1_stride, const float* __restrict__ g2,
                                                      const uint16_t* __restrict__ y, float slope,
                                                      int r, int gc, int dz_c,
                                                      uint16_t* __restrict__ dz) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t nvox = static_cast<int64_t>(r) * r * r;
  if (idx >= nvox * dz_c) return;
  const int c = static_cast<int>(idx % dz_c);
  const int v = static_cast<int>(idx / dz_c);
  float g = 0.0f;
  if (c < gc) {
    if (g1) g = g1[static_cast<int64_t>(v) * g1_stride + c];
    if (g2) {
      const int rc = r >> 1;
      const int x = v % r, yy = (v / r) % r, z = v / (r * r);
      const int p = ((z >> 1) * rc + (yy >> 1)) * rc + (x >> 1);
      g += g2[static_cast<int64_t>(p) * gc + c] * 0.125f;
    }
    if (y && !(bf2f(y[static_cast<int64_t>(v) * gc + c]) > 0.0f)) g *= slope;
  }
  dz[idx] = f2bf(g);
}

// act_bwd_kernel, 8 channels of one voxel per thread (gc and dz_c multiples of 8, g1_stride of 4,
// 16-byte aligned arrays): the same values from 16-byte loads, with one voxel index per 8 of them (the
// scalar kernel divides in 64 bits for each): 7.3 -> 5.9 us a launch over the layers.
__global__ void __launch_bounds__(256) act_bwd8_kernel(const float* __restrict__ g1, int g1_stride,
                                                       const float* __restrict__ g2,
                                                       const uint16_t* __restrict__ y, float slope,
                                                       int r, int gc, int dz_c,
                                                       uint16_t* __restrict__ dz) {
  const uint32_t c8n = static_cast<uint32_t>(dz_c) >> 3;
  const uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t nvox = static_cast<uint32_t>(r) * r * r;
  const uint32_t v = idx / c8n, c = 8u * (idx - v * c8n);
  if (v >= nvox) return;
  float g[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (c < static_cast<uint32_t>(gc)) {
    if (g1) {
      const float4* p = reinterpret_cast<const float4*>(g1 + static_cast<int64_t>(v) * g1_stride + c);
      const float4 a = p[0], b = p[1];
      g[0] = a.x; g[1] = a.y; g[2] = a.z; g[3] = a.w;
      g[4] = b.x; g[5] = b.y; g[6] = b.z; g[7] = b.w;
    }
    if (g2) {
      const uint32_t ur = static_cast<uint32_t>(r), rc = ur >> 1;
      const uint32_t row = v / ur, x = v - row * ur, z = row / ur, yy = row - z * ur;
      const int64_t q = ((z >> 1) * rc + (yy >> 1)) * rc + (x >> 1);
      const float4* p = reinterpret_cast<const float4*>(g2 + q * gc + c);
      const float4 a = p[0], b = p[1];
      g[0] += a.x * 0.125f; g[1] += a.y * 0.125f; g[2] += a.z * 0.125f; g[3] += a.w * 0.125f;
      g[4] += b.x * 0.125f; g[5] += b.y * 0.125f; g[6] += b.z * 0.125f; g[7] += b.w * 0.125f;
    }
    if (y) {
      const u32x4_t h = load16(y + static_cast<int64_t>(v) * gc + c);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint16_t b = static_cast<uint16_t>((k & 1) ? h[k >> 1] >> 16 : h[k >> 1] & 0xffffu);
        if (!(bf2f(b) > 0.0f)) g[k] *= slope;
      }
    }
  }
  u32x4_t out;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    out[k] = static_cast<uint32_t>(f2bf(g[2 * k])) | (static_cast<uint32_t>(f2bf(g[2 * k + 1])) << 16);
  *reinterpret_cast<u32x4_t*>(dz + static_cast<int64_t>(v) * dz_c + c) = out;
}

// Gradient of a nearest-upsampled input: ga[vc][c] = sum over the 8 children of
// dx[child][c] (c < ca; dx has stride cstride), in child order.
__global__ void __launch_bounds__(256) upsum_kernel(const float* __restrict__ dx, int r,
                                                    int cstride, int ca, float* __restrict__ ga) {
  const int rc = r >> 1;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= static_cast<int64_t>(rc) * rc * rc * ca) return;
  const int c = static_cast<int>(idx % ca);
  const int vc = static_cast<int>(idx / ca);
  const int X = vc % rc, Y = (vc / rc) % rc, Z = vc / (rc * rc);
  float s = 0.0f;
  for (int child = 0; child < 8; ++child) {
    const int z = 2 * Z + (child >> 2), y = 2 * Y + ((child >> 1) & 1), x = 2 * X + (child & 1);
    s += dx[static_cast<int64_t>((z * r + y) * r + x) * cstride + c];
  }
  ga[idx] = s;
}

__global__ void __launch_bounds__(256) f32_to_bf16_kernel(const float* __restrict__ x,
                                                          int64_t count,
                                                          uint16_t* __restrict__ y) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < count) y[i] = f2bf(x[i]);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

namespace pm {
namespace conv {

int rows_pad(int cout) { return (cout + 15) / 16 * 16; }
int kpad(int cin) { return (27 * cin + 31) / 32 * 32; }
int store_channels(int c) { return (c + 7) / 8 * 8; }

pm_status check_input(const uint16_t* xa, int ca, const uint16_t* xb, int cb, int r, int up,
                      const char* who) {
  PM_REQUIRE(xa, std::string(who) + ": null input");
  PM_REQUIRE(r >= 1 && r <= 512, std::string(who) + ": resolution must be in [1, 512]");
  PM_REQUIRE(ca > 0 && ca % 8 == 0 && cb >= 0 && cb % 8 == 0 && ca + cb <= 1024,
             std::string(who) + ": channel counts must be multiples of 8 (ca > 0, total <= 1024)");
  PM_REQUIRE(cb == 0 || xb, std::string(who) + ": cb > 0 needs xb");
  PM_REQUIRE(!up || r % 2 == 0, std::string(who) + ": upsampled input needs an even resolution");
  PM_REQUIRE(aligned16(xa) && (!xb || aligned16(xb)),
             std::string(who) + ": inputs must be 16-byte aligned");
  return PM_OK;
}

// Launch shape of a forward convolution: column groups of 16*NB output channels and
// reduction splits so that small grids (the network's coarse levels) still spread over the
// chip. Split-K needs float32 scratch for the raw sums (fwd_scratch_floats).
struct FwdPlan {
  int nb = 8, groups = 1, ksplit = 1, kc_per = 1;
};

FwdPlan fwd_plan(int nvox, int rows, int kpad_, bool allow_split) {
  constexpr int64_t kTargetWaves = 2048;
  FwdPlan p;
  const int64_t vox_waves = (nvox + 63) / 64;
  p.nb = std::min(8, rows / 16);
  while (p.nb > 1 && vox_waves * ((rows + 16 * p.nb - 1) / (16 * p.nb)) < kTargetWaves) p.nb /= 2;
  if (p.nb == 3) p.nb = 2;
  p.groups = (rows + 16 * p.nb - 1) / (16 * p.nb);
  const int kchunks = kpad_ / 32;
  const int64_t waves = vox_waves * p.groups;
  if (allow_split && waves < kTargetWaves) {
    int64_t want = kTargetWaves / std::max<int64_t>(1, waves);
    want = std::min<int64_t>(want, std::max(1, kchunks / 4));
    want = std::min<int64_t>(want, 32);
    p.ksplit = static_cast<int>(std::max<int64_t>(1, want));
  }
  p.kc_per = (kchunks + p.ksplit - 1) / p.ksplit;
  p.ksplit = (kchunks + p.kc_per - 1) / p.kc_per;
  return p;
}

// Input channel counts that conv_tile_kernel is built for. A tile takes 400 * (2 * channels + 16)
// bytes of LDS: 108,800 for 128, 83,200 for each half of 192.
bool tile_fits(int cin) {
  switch (cin) {
    case 8: case 16: case 32: case 48: case 64: case 96: case 128: case 192: return true;
    default: return false;
  }
}

template <int CIN, int S>
void launch_tile(const ConvTileArgs& t, int nb, dim3 grid, hipStream_t s) {
  constexpr size_t lds = static_cast<size_t>(kHaloVox) * (2 * CIN / S + 16);
  static_assert(lds <= 160 * 1024, "the tile fits the LDS");
  if (nb == 1) conv_tile_kernel<CIN, 1, S><<<grid, 256, lds, s>>>(t);
  else if (nb == 2) conv_tile_kernel<CIN, 2, S><<<grid, 256, lds, s>>>(t);
  else conv_tile_kernel<CIN, 3, S><<<grid, 256, lds, s>>>(t);
}

pm_status fwd_tile(const ConvFwdArgs& a, const char* timer, hipStream_t s) {
  const int tx = (a.r + 7) / 8, tz = (a.r + 1) / 2;
  ConvTileArgs t;
  t.c = a;
  t.c.partial = nullptr;
  t.dt = pm::make_fast_div(static_cast<uint32_t>(tx));
  const int blocks = a.rows / 16;
  const int64_t tiles = static_cast<int64_t>(tx) * tx * tz;
  // column blocks per workgroup: as many as leave two workgroups per CU
  int nb = std::min(3, blocks);
  while (nb > 1 && tiles * ((blocks + nb - 1) / nb) < 512) --nb;
  const dim3 grid(static_cast<unsigned>(tiles), static_cast<unsigned>((blocks + nb - 1) / nb));
  const double flops = 2.0 * 27.0 * a.cin * a.cout * static_cast<double>(a.r) * a.r * a.r;
  PM_TIMED(timer, flops, s);
  switch (a.cin) {
    case 8: launch_tile<8, 1>(t, nb, grid, s); break;
    case 16: launch_tile<16, 1>(t, nb, grid, s); break;
    case 32: launch_tile<32, 1>(t, nb, grid, s); break;
    case 48: launch_tile<48, 1>(t, nb, grid, s); break;
    case 64: launch_tile<64, 1>(t, nb, grid, s); break;
    case 96: launch_tile<96, 3>(t, nb, grid, s); break;
    case 128: launch_tile<128, 1>(t, nb, grid, s); break;
    default: launch_tile<192, 2>(t, nb, grid, s); break;
  }
  PM_CHECK_LAUNCH("conv_tile_kernel");
  return PM_OK;
}

// Scratch of conv_fwd_kernel's split, whether or not it serves these widths.
int64_t split_scratch_floats(int cin, int cout, int r) {
  const int64_t nvox = static_cast<int64_t>(r) * r * r;
  const FwdPlan p = fwd_plan(static_cast<int>(nvox), rows_pad(cout), kpad(cin), true);
  return p.ksplit > 1 ? p.ksplit * nvox * rows_pad(cout) : 0;
}

int64_t fwd_scratch_floats(int cin, int cout, int r) {
  return tile_fits(cin) ? 0 : split_scratch_floats(cin, cout, r);
}

pm_status fwd(const uint16_t* xa, int ca, const uint16_t* xb, int cb, int r, int up,
              const uint16_t* wp, const float* bias, int cout, int act, float slope, uint16_t* y,
              float* y32, const char* timer, hipStream_t s, float* scratch,
              int64_t scratch_floats) {
  pm_status st;
  if ((st = check_input(xa, ca, xb, cb, r, up, "pm_conv3d_fwd_bf16"))) return st;
  PM_REQUIRE(wp && aligned16(wp), "pm_conv3d_fwd_bf16: weights null or not 16-byte aligned");
  PM_REQUIRE(cout >= 1 && cout <= 1024, "pm_conv3d_fwd_bf16: cout must be in [1, 1024]");
  PM_REQUIRE(y || y32, "pm_conv3d_fwd_bf16: no output");
  ConvFwdArgs a;
  a.xa = xa;
  a.xb = cb ? xb : nullptr;
  a.ca = ca;
  a.cb = cb;
  a.cin = ca + cb;
  a.r = r;
  a.ra = up ? r / 2 : r;
  a.up = up ? 1 : 0;
  a.w = wp;
  a.kpad = kpad(a.cin);
  a.kreal = 27 * a.cin;
  a.rows = rows_pad(cout);
  a.bias = bias;
  a.cout = cout;
  a.cout_st = store_channels(cout);
  a.act = act ? 1 : 0;
  a.slope = slope;
  a.y = y;
  a.y32 = y32;
  const int nvox = r * r * r;
  if (tile_fits(a.cin)) return fwd_tile(a, timer, s);
  FwdPlan p = fwd_plan(nvox, a.rows, a.kpad, scratch != nullptr);
  if (p.ksplit > 1 && static_cast<int64_t>(p.ksplit) * nvox * a.rows > scratch_floats)
    p = fwd_plan(nvox, a.rows, a.kpad, false);
  a.kc_per = p.kc_per;
  a.partial = p.ksplit > 1 ? scratch : nullptr;
  const dim3 grid(static_cast<unsigned>((nvox + 255) / 256), static_cast<unsigned>(p.groups),
                  static_cast<unsigned>(p.ksplit));
  const double flops = 2.0 * 27.0 * a.cin * cout * static_cast<double>(nvox);
  PM_TIMED(timer, flops, s);
  switch (p.nb) {
    case 1: conv_fwd_kernel<1><<<grid, 256, 0, s>>>(a); break;
    case 2: conv_fwd_kernel<2><<<grid, 256, 0, s>>>(a); break;
    case 4: conv_fwd_kernel<4><<<grid, 256, 0, s>>>(a); break;
    default: conv_fwd_kernel<8><<<grid, 256, 0, s>>>(a); break;
  }
  PM_CHECK_LAUNCH("conv_fwd_kernel");
  if (p.ksplit > 1) {
    const int64_t total = static_cast<int64_t>(nvox) * a.cout_st;
    conv_epilogue_kernel<<<pm::blocks_for(total), 256, 0, s>>>(
        scratch, p.ksplit, nvox, a.rows, bias, cout, a.cout_st, a.act, slope, y, y32);
    PM_CHECK_LAUNCH("conv_epilogue_kernel");
  }
  return PM_OK;
}

int64_t wgrad_partial_floats(int cin, int cout, int r) {
  int splits, chunks;
  wgrad_plan(cin, cout, r, &splits, &chunks);
  const int kcols = (kpad(cin) + 63) / 64 * 64;
  const int rows = rows_pad(store_channels(cout));
  return static_cast<int64_t>(splits) * rows * (kcols + 1);  // and the channel sums
}

// About 1024 workgroups, 4 per CU: with 2048 the stages are too few to hide their loads and the
// fold reads twice the partial sums (weight gradients of a 4-pair batch 1.95 ms against 1.88),
// with 512 too few loads are in flight (2.29 ms).
void wgrad_plan(int cin, int cout, int r, int* splits, int* chunks_per_split) {
  (void)cout;
  const int64_t nvox = static_cast<int64_t>(r) * r * r;
  const int64_t nchunks = (nvox + 31) / 32;
  const int kgroups = (kpad(cin) + 63) / 64;
  int64_t want = std::max<int64_t>(1, 1024 / kgroups);
  want = std::min<int64_t>(want, nchunks);
  const int64_t per = (nchunks + want - 1) / want;
  *chunks_per_split = static_cast<int>(per);
  *splits = static_cast<int>((nchunks + per - 1) / per);
}

pm_status wgrad(const uint16_t* xa, int ca, const uint16_t* xb, int cb, int r, int up,
                const uint16_t* dz, int cout, float* dw, float* db, int accumulate,
                float* partial, int64_t partial_floats, const char* timer, hipStream_t s) {
  pm_status st;
  if ((st = check_input(xa, ca, xb, cb, r, up, "pm_conv3d_bwd_weight_bf16"))) return st;
  PM_REQUIRE(dz && aligned16(dz) && dw && partial,
             "pm_conv3d_bwd_weight_bf16: null or misaligned pointer");
  PM_REQUIRE(cout >= 1 && cout <= 128, "pm_conv3d_bwd_weight_bf16: cout must be in [1, 128]");
  const int cin = ca + cb;
  const int dz_c = store_channels(cout);
  PM_REQUIRE((dz_c & (dz_c - 1)) == 0,
             "pm_conv3d_bwd_weight_bf16: cout must round up (to a multiple of 8) to a power of two");
  PM_REQUIRE(partial_floats >= wgrad_partial_floats(cin, cout, r),
             "pm_conv3d_bwd_weight_bf16: partial buffer too small");
  int splits, chunks;
  wgrad_plan(cin, cout, r, &splits, &chunks);
  ConvWgradArgs a;
  a.xa = xa;
  a.xb = cb ? xb : nullptr;
  a.ca = ca;
  a.cb = cb;
  a.cin = cin;
  a.r = r;
  a.ra = up ? r / 2 : r;
  a.up = up ? 1 : 0;
  a.dz = dz;
  a.dz_c = dz_c;
  a.kreal = 27 * cin;
  a.nvox = r * r * r;
  a.chunks_per_split = chunks;
  a.partial = partial;
  a.kcols = (kpad(cin) + 63) / 64 * 64;
  const int nr = std::max(1, rows_pad(dz_c) / 16);  // 1, 2, 4 or 8 (dz_c is 8..128)
  const int rows = 16 * nr;
  a.partial_b = db ? partial + static_cast<int64_t>(splits) * rows * a.kcols : nullptr;
  const dim3 grid(static_cast<unsigned>(a.kcols / 64), static_cast<unsigned>(splits));
  {
    const double flops = 2.0 * 27.0 * cin * cout * static_cast<double>(a.nvox);
    PM_TIMED(timer, flops, s);
    switch (nr) {
      case 1: conv_wgrad_kernel<1, 128><<<grid, 256, 0, s>>>(a); break;
      case 2: conv_wgrad_kernel<2, 128><<<grid, 256, 0, s>>>(a); break;
      case 4: conv_wgrad_kernel<4, 64><<<grid, 256, 0, s>>>(a); break;
      default: conv_wgrad_kernel<8, 64><<<grid, 256, 0, s>>>(a); break;
    }
    PM_CHECK_LAUNCH("conv_wgrad_kernel");
  }
  const dim3 fold(static_cast<unsigned>(a.kcols / 64), static_cast<unsigned>(cout + (db ? 1 : 0)));
  wgrad_fold_kernel<<<fold, 64 * kFoldWaves, 0, s>>>(partial, a.partial_b, splits, cout, rows,
                                                     a.kcols, cin, dw, db, accumulate);
  PM_CHECK_LAUNCH("wgrad_fold_kernel");
  return PM_OK;
}

pm_status pack(const float* w, int cout, int cin, int transpose, uint16_t* wp, hipStream_t s) {
  PM_REQUIRE(w && wp, "pm_conv3d_pack_weights: null pointer");
  PM_REQUIRE(cout >= 1 && cout <= 1024 && cin >= 1 && cin <= 1024,
             "pm_conv3d_pack_weights: channel counts out of range");
  int rows, kp, cin_eff;
  if (!transpose) {
    rows = rows_pad(cout);
    cin_eff = cin;
    kp = kpad(cin);
  } else {
    rows = rows_pad(cin);
    cin_eff = store_channels(cout);
    kp = kpad(cin_eff);
  }
  const int64_t total = static_cast<int64_t>(rows) * kp;
  pack_weights_kernel<<<pm::blocks_for(total), 256, 0, s>>>(w, cout, cin, transpose, cin_eff, rows,
                                                            kp, wp);
  PM_CHECK_LAUNCH("pack_weights_kernel");
  return PM_OK;
}

int64_t packed_elems(int cout, int cin, int transpose) {
  if (!transpose) return static_cast<int64_t>(rows_pad(cout)) * kpad(cin);
  return static_cast<int64_t>(rows_pad(cin)) * kpad(store_channels(cout));
}

pm_status pool2(const uint16_t* x, int r, int c, uint16_t* y, hipStream_t s) {
  PM_REQUIRE(x && y && aligned16(x) && aligned16(y), "pm_pool2_bf16: null or misaligned pointer");
  PM_REQUIRE(r >= 2 && r % 2 == 0 && c % 8 == 0 && c > 0, "pm_pool2_bf16: bad shape");
  const int64_t total = static_cast<int64_t>(r / 2) * (r / 2) * (r / 2) * (c / 8);
  PM_TIMED("net.pool", 2.0 * c * (static_cast<double>(r) * r * r + total * 8.0 / c), s);
  pool2_kernel<<<pm::blocks_for(total), 256, 0, s>>>(x, r, c, y);
  PM_CHECK_LAUNCH("pool2_kernel");
  return PM_OK;
}

pm_status act_bwd(const float* g1, int g1_stride, const float* g2, const uint16_t* y, float slope,
                  int r, int gc, int dz_c, uint16_t* dz, hipStream_t s) {
  PM_REQUIRE(dz, "pm_act_bwd_bf16: null output");
  PM_REQUIRE(gc >= 1 && dz_c >= gc && r >= 1, "pm_act_bwd_bf16: bad shape");
  PM_REQUIRE(!g2 || r % 2 == 0, "pm_act_bwd_bf16: pooled gradient needs an even resolution");
  const int64_t total = static_cast<int64_t>(r) * r * r * dz_c;
  PM_TIMED("net.act_bwd", 6.0 * static_cast<double>(total), s);
  const bool wide = gc % 8 == 0 && dz_c % 8 == 0 && total < (int64_t(1) << 33) &&
                    (!g1 || (g1_stride % 4 == 0 && aligned16(g1))) &&
                    (!g2 || aligned16(g2)) && (!y || aligned16(y)) && aligned16(dz);
  if (wide)
    act_bwd8_kernel<<<pm::blocks_for(total / 8), 256, 0, s>>>(g1, g1_stride, g2, y, slope, r, gc,
                                                              dz_c, dz);
  else
    act_bwd_kernel<<<pm::blocks_for(total), 256, 0, s>>>(g1, g1_stride, g2, y, slope, r, gc, dz_c,
                                                         dz);
  PM_CHECK_LAUNCH("act_bwd_kernel");
  return PM_OK;
}

pm_status upsum(const float* dx, int r, int cstride, int ca, float* ga, hipStream_t s) {
  PM_REQUIRE(dx && ga, "pm_upsum_f32: null pointer");
  PM_REQUIRE(r % 2 == 0 && ca >= 1 && cstride >= ca, "pm_upsum_f32: bad shape");
  const int64_t total = static_cast<int64_t>(r / 2) * (r / 2) * (r / 2) * ca;
  PM_TIMED("net.upsum", 36.0 * static_cast<double>(total), s);
  upsum_kernel<<<pm::blocks_for(total), 256, 0, s>>>(dx, r, cstride, ca, ga);
  PM_CHECK_LAUNCH("upsum_kernel");
  return PM_OK;
}

pm_status to_bf16(const float* x, int64_t count, uint16_t* y, hipStream_t s) {
  PM_REQUIRE(x && y && count >= 0, "pm_f32_to_bf16: bad argument");
  if (count == 0) return PM_OK;
  f32_to_bf16_kernel<<<pm::blocks_for(count), 256, 0, s>>>(x, count, y);
  PM_CHECK_LAUNCH("f32_to_bf16_kernel");
  return PM_OK;
}

}  // namespace conv
}  // namespace pm

extern "C" {

pm_status pm_conv3d_packed_size(int32_t cout, int32_t cin, int32_t transpose, int64_t* elems) {
  PM_REQUIRE(elems && cout >= 1 && cin >= 1, "pm_conv3d_packed_size: bad argument");
  *elems = pm::conv::packed_elems(cout, cin, transpose);
  return PM_OK;
}

pm_status pm_conv3d_pack_weights(const float* w, int32_t cout, int32_t cin, int32_t transpose,
                                 uint16_t* packed, hipStream_t s) {
  pm::clear_error();
  return pm::conv::pack(w, cout, cin, transpose, packed, s);
}

pm_status pm_conv3d_scratch_size(int32_t cin, int32_t cout, int32_t r, int64_t* floats) {
  PM_REQUIRE(floats && cin >= 1 && cout >= 1 && r >= 1, "pm_conv3d_scratch_size: bad argument");
  *floats = std::max(pm::conv::split_scratch_floats(cin, cout, r),
                     pm::conv::split_scratch_floats(pm::conv::store_channels(cout), cin, r));
  return PM_OK;
}

pm_status pm_conv3d_fwd_bf16(const uint16_t* xa, int32_t ca, const uint16_t* xb, int32_t cb,
                             int32_t r, int32_t up_a, const uint16_t* packed, const float* bias,
                             int32_t cout, int32_t act, float slope, uint16_t* y, float* y32,
                             float* scratch, int64_t scratch_floats, hipStream_t s) {
  pm::clear_error();
  return pm::conv::fwd(xa, ca, xb, cb, r, up_a, packed, bias, cout, act, slope, y, y32,
                       "net.conv_fwd", s, scratch, scratch ? scratch_floats : 0);
}

pm_status pm_conv3d_bwd_data_bf16(const uint16_t* dz, int32_t cout, int32_t r,
                                  const uint16_t* packed_t, int32_t cin, float* dx,
                                  float* scratch, int64_t scratch_floats, hipStream_t s) {
  pm::clear_error();
  PM_REQUIRE(dz && packed_t && dx, "pm_conv3d_bwd_data_bf16: null pointer");
  return pm::conv::fwd(dz, pm::conv::store_channels(cout), nullptr, 0, r, 0, packed_t, nullptr,
                       cin, 0, 0.0f, nullptr, dx, "net.conv_bwd_data", s, scratch,
                       scratch ? scratch_floats : 0);
}

pm_status pm_conv3d_wgrad_partial_size(int32_t cin, int32_t cout, int32_t r, int64_t* floats) {
  PM_REQUIRE(floats && cin >= 1 && cout >= 1 && r >= 1, "pm_conv3d_wgrad_partial_size: bad argument");
  *floats = pm::conv::wgrad_partial_floats(cin, cout, r);
  return PM_OK;
}

pm_status pm_conv3d_bwd_weight_bf16(const uint16_t* xa, int32_t ca, const uint16_t* xb,
                                    int32_t cb, int32_t r, int32_t up_a, const uint16_t* dz,
                                    int32_t cout, float* dw, float* db, int32_t accumulate,
                                    float* partial, int64_t partial_floats, hipStream_t s) {
  pm::clear_error();
  return pm::conv::wgrad(xa, ca, xb, cb, r, up_a, dz, cout, dw, db, accumulate, partial,
                         partial_floats, "net.conv_bwd_weight", s);
}

pm_status pm_pool2_bf16(const uint16_t* x, int32_t r, int32_t c, uint16_t* y, hipStream_t s) {
  pm::clear_error();
  return pm::conv::pool2(x, r, c, y, s);
}

pm_status pm_act_bwd_bf16(const float* g1, int32_t g1_stride, const float* g2, const uint16_t* y,
                          float slope, int32_t r, int32_t gc, int32_t dz_c, uint16_t* dz,
                          hipStream_t s) {
  pm::clear_error();
  return pm::conv::act_bwd(g1, g1_stride, g2, y, slope, r, gc, dz_c, dz, s);
}

pm_status pm_upsum_f32(const float* dx, int32_t r, int32_t cstride, int32_t ca, float* ga,
                       hipStream_t s) {
  pm::clear_error();
  return pm::conv::upsum(dx, r, cstride, ca, ga, s);
}

pm_status pm_f32_to_bf16(const float* x, int64_t count, uint16_t* y, hipStream_t s) {
  pm::clear_error();
  return pm::conv::to_bf16(x, count, y, s);
}

}  // extern "C"
