// Device 2D mass projection (reference viz/project.py:26-83): nearest-bin (NGP) mass per
// bin over two in-plane axes, the third projected out; out-of-extent particles dropped.
//
// The reference scatters with float atomics, so its sums depend on the arrival order. Here
// each particle's mass is converted to a fixed-point integer (scale 2^s chosen from the
// largest mass so that any sum of up to 2^28 particles fits in 63 bits) and accumulated with
// 64-bit integer atomics, which commute: the image is identical run to run, and the only
// error is the quantization of each mass (relative <= 2^-34 of the largest mass).
//
// Integer sums commute, so where they are added is free to choose. Two paths give the same
// image bit for bit:
//   direct  one global 64-bit atomic per particle: few launches, but the atomics of a
//           concentrated image queue up at its hot bins (3.0 ms for 10M particles of a
//           collision on 512^2 bins, 40 GB/s of the 120 MB read);
//   tiled   the particles are partitioned by 64 x 64-bin image tile first (count, scan,
//           scatter of 8-byte records), then every workgroup sums one chunk of records in
//           LDS and adds its non-zero bins to the image once. The same 10M particles take
//           117 us (cell order; 130 in random order): count 32, scan 8, scatter 42, sums 30,
//           unscale 5. It reads the particles twice and writes and reads 8 bytes for each;
//           the bin arithmetic (two IEEE divisions) and the LDS ranks bound the first two,
//           same-bin LDS atomics the third.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "pm_common.h"
#include "pm_timing.h"

namespace {

// Largest value over the workgroup (256 threads), in every thread. Uniform control flow only.
__device__ __forceinline__ unsigned int block_max(unsigned int m) {
  __shared__ unsigned int s[4];
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned int o = __shfl_xor(m, off, 64);
    m = o > m ? o : m;
  }
  if ((threadIdx.x & 63u) == 0) s[threadIdx.x >> 6] = m;
  __syncthreads();
  for (int w = 0; w < 4; ++w) m = s[w] > m ? s[w] : m;
  return m;
}

// First launch of the direct path: clears acc[0..cells] and leaves each workgroup's largest
// mass (bit patterns: masses are non-negative, so their float bits order like the values) in
// maxima[blockIdx.x]; the scatter's workgroups reduce those, so the maximum costs no launch of
// its own (20,000 particles on 256 bins 15.6 us a frame with four launches, 14.2 with three;
// 190,000 on 512 24.5 -> 16.1).
constexpr int kMaxima = 1024;
__global__ void __launch_bounds__(256) clear_max_kernel(const float* __restrict__ mass, int64_t n,
                                                        unsigned long long* __restrict__ acc,
                                                        int64_t cells,
                                                        unsigned int* __restrict__ maxima) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t step = static_cast<int64_t>(gridDim.x) * blockDim.x;
  unsigned int m = 0u;
  for (int64_t i = t; i < n; i += step) {
    const float v = mass[i];
    const unsigned int b = v > 0.0f ? __float_as_uint(v) : 0u;
    m = b > m ? b : m;
  }
  for (int64_t i = t; i <= cells; i += step) acc[i] = 0ull;
  m = block_max(m);
  if (threadIdx.x == 0) maxima[blockIdx.x] = m;
}

// scale exponent: largest mass * 2^s < 2^34 (s from the max mass's binary exponent)
__device__ __forceinline__ int scale_exp(unsigned int maxbits) {
  if (maxbits == 0u) return 0;
  const int e = static_cast<int>((maxbits >> 23) & 0xffu) - 127;  // max in [2^e, 2^(e+1))
  return 33 - e;
}

// Bin of a particle, or false where it is dropped. The range test on the float value also
// rejects NaN and values beyond int range.
__device__ __forceinline__ bool bin_of(float a, float b, float lo_a, float lo_b, float binw_a,
                                       float binw_b, int bins, int& ia, int& ib) {
  const float fa = floorf((a - lo_a) / binw_a);
  const float fb = floorf((b - lo_b) / binw_b);
  if (!(fa >= 0.0f && fa < static_cast<float>(bins) && fb >= 0.0f && fb < static_cast<float>(bins)))
    return false;
  ia = static_cast<int>(fa);
  ib = static_cast<int>(fb);
  return true;
}

// Fixed-point mass; zero, negative or non-finite masses add nothing.
__device__ __forceinline__ unsigned long long fixed_mass(float m, unsigned int maxbits) {
  const double q = ldexp(static_cast<double>(m), scale_exp(maxbits));
  if (!(q > 0.0 && q < 1.8e16)) return 0ull;
  return static_cast<unsigned long long>(llrint(q));
}

__global__ void __launch_bounds__(256) project_kernel(const float* __restrict__ pa,
                                                      const float* __restrict__ pb,
                                                      const float* __restrict__ mass, int64_t n,
                                                      float lo_a, float lo_b, float binw_a,
                                                      float binw_b, int bins,
                                                      const unsigned int* __restrict__ maxima,
                                                      int nmax,
                                                      unsigned int* __restrict__ maxbits,
                                                      unsigned long long* __restrict__ acc) {
  unsigned int top = 0u;
  for (int t = threadIdx.x; t < nmax; t += blockDim.x) top = maxima[t] > top ? maxima[t] : top;
  top = block_max(top);
  if (blockIdx.x == 0 && threadIdx.x == 0) *maxbits = top;  // for unscale_kernel
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    int ia, ib;
    if (!bin_of(pa[i], pb[i], lo_a, lo_b, binw_a, binw_b, bins, ia, ib)) continue;
    const unsigned long long q = fixed_mass(mass[i], top);
    if (q) atomicAdd(&acc[static_cast<int64_t>(ia) * bins + ib], q);
  }
}

// ---- tiled path ------------------------------------------------------------------------

constexpr int kTileBits = 6;                     // 64 x 64 bins: 32 KB of LDS sums
constexpr int kTileSide = 1 << kTileBits;
constexpr int kTileBins = kTileSide * kTileSide;
constexpr int kMaxTiles = 256;                   // bins <= 1024
constexpr int kGroup = 4096;                     // particles per counting / scatter workgroup
constexpr int kChunk = 8192;                     // records per summing workgroup
constexpr int64_t kSlab = int64_t{1} << 24;      // records held at once (128 MiB of scratch)

// Adds one to counter[t] for every lane with t >= 0 and returns the lane's old value. Cell
// ordered particles put a whole wave into one tile: that wave makes a single LDS atomic (64
// same-address ones would be served one after the other).
__device__ __forceinline__ unsigned wave_add(unsigned* counter, int t) {
  const unsigned long long live = __ballot(t >= 0);
  if (!live) return 0u;
  const int src = __ffsll(live) - 1;
  const int t0 = __builtin_amdgcn_readlane(t, src);
  if (__ballot(t >= 0 && t == t0) == live) {
    const int lane = threadIdx.x & 63;
    unsigned base = 0u;
    if (lane == src) base = atomicAdd(&counter[t0], static_cast<unsigned>(__popcll(live)));
    base = __builtin_amdgcn_readlane(base, src);
    return base + static_cast<unsigned>(__popcll(live & ((1ull << lane) - 1ull)));
  }
  return t >= 0 ? atomicAdd(&counter[t], 1u) : 0u;
}

struct ProjectArgs {
  const float* pa;
  const float* pb;
  const float* mass;
  int64_t n;
  float lo_a, lo_b, binw_a, binw_b;
  int bins, tiles_b, tiles;
  int groups;                  // counting workgroups: ceil(n / kGroup)
  unsigned* group_max;         // [groups] largest mass bits
  unsigned* maxbits;
  unsigned* hist;              // [tiles][groups] counts, then exclusive prefixes per slab
  unsigned* totals;            // [tiles] records of the slab
  unsigned long long* records;
  unsigned long long* acc;     // [bins][bins]
};

__device__ __forceinline__ int tile_of(const ProjectArgs& a, float x, float y, int& local) {
  int ia, ib;
  if (!bin_of(x, y, a.lo_a, a.lo_b, a.binw_a, a.binw_b, a.bins, ia, ib)) return -1;
  local = ((ia & (kTileSide - 1)) << kTileBits) | (ib & (kTileSide - 1));
  return (ia >> kTileBits) * a.tiles_b + (ib >> kTileBits);
}

// Per group of particles: records per tile and the largest mass; also clears the image sums.
__global__ void __launch_bounds__(256) tile_count_kernel(ProjectArgs a) {
  __shared__ unsigned cnt[kMaxTiles];
  __shared__ unsigned smax[4];
  const int tid = threadIdx.x;
  const int64_t cells = static_cast<int64_t>(a.bins) * a.bins;
  for (int64_t c = static_cast<int64_t>(blockIdx.x) * 256 + tid; c < cells;
       c += static_cast<int64_t>(gridDim.x) * 256)
    a.acc[c] = 0ull;
  cnt[tid] = 0u;
  __syncthreads();
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kGroup;
  unsigned m = 0u;
#pragma unroll 4
  for (int r = 0; r < kGroup / 256; ++r) {
    const int64_t i = base + r * 256 + tid;
    int t = -1, local;
    if (i < a.n) {
      const float v = a.mass[i];
      t = tile_of(a, a.pa[i], a.pb[i], local);
      const unsigned b = v > 0.0f ? __float_as_uint(v) : 0u;
      m = b > m ? b : m;
    }
    wave_add(cnt, t);
  }
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned o = __shfl_down(m, off);
    m = o > m ? o : m;
  }
  if ((tid & 63) == 0) smax[tid >> 6] = m;
  __syncthreads();
  if (tid < a.tiles) a.hist[static_cast<int64_t>(tid) * a.groups + blockIdx.x] = cnt[tid];
  if (tid == 0) {
    for (int w = 1; w < 4; ++w) m = smax[w] > m ? smax[w] : m;
    a.group_max[blockIdx.x] = m;
  }
}

// One workgroup per tile: exclusive prefix of its counts over the slab's groups [g0, g1) and
// their total; workgroup 0 also folds the largest mass over all groups.
__global__ void __launch_bounds__(256) tile_scan_kernel(ProjectArgs a, int g0, int g1) {
  __shared__ unsigned s[256];
  const int tid = threadIdx.x;
  unsigned* h = a.hist + static_cast<int64_t>(blockIdx.x) * a.groups;
  const int per = (g1 - g0 + 255) / 256;
  const int b = min(g1, g0 + tid * per), e = min(g1, b + per);
  unsigned sum = 0u;
  for (int g = b; g < e; ++g) sum += h[g];
  s[tid] = sum;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const unsigned v = tid >= off ? s[tid - off] : 0u;
    __syncthreads();
    s[tid] += v;
    __syncthreads();
  }
  unsigned run = s[tid] - sum;
  for (int g = b; g < e; ++g) {
    const unsigned c = h[g];
    h[g] = run;
    run += c;
  }
  if (tid == 255) a.totals[blockIdx.x] = s[255];
  if (blockIdx.x == 0) {
    __syncthreads();
    unsigned m = 0u;
    for (int g = tid; g < a.groups; g += 256) m = max(m, a.group_max[g]);
    s[tid] = m;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
      if (tid < off) s[tid] = max(s[tid], s[tid + off]);
      __syncthreads();
    }
    if (tid == 0) *a.maxbits = s[0];
  }
}

// start[t] = first record of tile t (exclusive prefix of totals), start[kMaxTiles] = all;
// kMaxTiles threads take part.
__device__ __forceinline__ void tile_starts(const ProjectArgs& a, unsigned* start) {
  const int tid = threadIdx.x;
  const unsigned mine = tid < a.tiles ? a.totals[tid] : 0u;
  if (tid < kMaxTiles) start[tid + 1] = mine;
  if (tid == 0) start[0] = 0u;
  __syncthreads();
  for (int off = 1; off < kMaxTiles; off <<= 1) {
    const unsigned v = (tid < kMaxTiles && tid >= off) ? start[tid + 1 - off] : 0u;
    __syncthreads();
    if (tid < kMaxTiles) start[tid + 1] += v;
    __syncthreads();
  }
}

// Scatters the slab's records (fixed-point mass << 12 | bin in tile; the mass is < 2^35) to
// their tiles. The order inside a tile does not matter: the sums are integers.
__global__ void __launch_bounds__(256) tile_scatter_kernel(ProjectArgs a, int g0) {
  __shared__ unsigned start[kMaxTiles + 1];
  __shared__ unsigned cursor[kMaxTiles];
  const int tid = threadIdx.x;
  const int g = g0 + static_cast<int>(blockIdx.x);
  tile_starts(a, start);
  cursor[tid] = tid < a.tiles ? start[tid] + a.hist[static_cast<int64_t>(tid) * a.groups + g] : 0u;
  const unsigned maxbits = *a.maxbits;
  __syncthreads();
  const int64_t base = static_cast<int64_t>(g) * kGroup;
#pragma unroll 4
  for (int r = 0; r < kGroup / 256; ++r) {
    const int64_t i = base + r * 256 + tid;
    int t = -1, local = 0;
    unsigned long long q = 0ull;
    if (i < a.n) {
      const float v = a.mass[i];
      t = tile_of(a, a.pa[i], a.pb[i], local);
      q = fixed_mass(v, maxbits);
    }
    const unsigned at = wave_add(cursor, t);
    if (t >= 0) a.records[at] = (q << (2 * kTileBits)) | static_cast<unsigned>(local);
  }
}

// One chunk of records per workgroup, tile by tile: bin sums in LDS, then one global atomic
// per non-zero bin.
__global__ void __launch_bounds__(512) tile_sum_kernel(ProjectArgs a) {
  __shared__ unsigned start[kMaxTiles + 1];
  __shared__ unsigned long long sum[kTileBins];
  const int tid = threadIdx.x;
  tile_starts(a, start);
  const unsigned all = start[kMaxTiles];
  const unsigned c0 = blockIdx.x * static_cast<unsigned>(kChunk);
  if (c0 >= all) return;
  const unsigned c1 = min(all, c0 + static_cast<unsigned>(kChunk));
  int t = 0;  // the tile of record c0: the last one that starts at or before it
  for (int step = kMaxTiles / 2; step > 0; step >>= 1)
    if (start[t + step] <= c0) t += step;
  for (int b = tid; b < kTileBins; b += 512) sum[b] = 0ull;
  __syncthreads();
  for (unsigned at = c0; at < c1;) {
    while (start[t + 1] <= at) ++t;  // empty tiles
    const unsigned end = min(c1, start[t + 1]);
    for (unsigned i = at + tid; i < end; i += 512) {
      const unsigned long long rec = a.records[i];
      const unsigned long long q = rec >> (2 * kTileBits);
      if (q) atomicAdd(&sum[rec & (kTileBins - 1)], q);
    }
    __syncthreads();
    const int a0 = (t / a.tiles_b) << kTileBits, b0 = (t % a.tiles_b) << kTileBits;
    for (int b = tid; b < kTileBins; b += 512) {
      const unsigned long long v = sum[b];
      if (v) {
        atomicAdd(&a.acc[static_cast<int64_t>(a0 + (b >> kTileBits)) * a.bins + b0 +
                         (b & (kTileSide - 1))],
                  v);
        sum[b] = 0ull;
      }
    }
    __syncthreads();
    at = end;
  }
}

__global__ void __launch_bounds__(256) unscale_kernel(const unsigned long long* __restrict__ acc,
                                                      int64_t count,
                                                      const unsigned int* __restrict__ maxbits,
                                                      float* __restrict__ img) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < count)
    img[i] = static_cast<float>(ldexp(static_cast<double>(acc[i]), -scale_exp(*maxbits)));
}

}  // namespace

namespace {

// Byte offsets of the tiled path's scratch.
struct TiledLayout {
  int tiles_b, tiles, groups;
  int64_t acc, records, hist, group_max, totals, maxbits, bytes;
};

TiledLayout tiled_layout(int64_t n, int bins) {
  TiledLayout l;
  l.tiles_b = (bins + kTileSide - 1) / kTileSide;
  l.tiles = l.tiles_b * l.tiles_b;
  l.groups = static_cast<int>((n + kGroup - 1) / kGroup);
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t here = at;
    at += (bytes + 15) / 16 * 16;
    return here;
  };
  l.acc = take(8 * static_cast<int64_t>(bins) * bins);
  l.records = take(8 * std::min(n, kSlab));
  l.hist = take(4 * static_cast<int64_t>(l.tiles) * l.groups);
  l.group_max = take(4 * static_cast<int64_t>(l.groups));
  l.totals = take(4 * kMaxTiles);
  l.maxbits = take(4);
  l.bytes = at;
  return l;
}

// The direct path's cost is the queue at the hottest bins, which shortens as the bins get
// smaller; the tiled path costs 35-70 us up to a million particles, more of it the more tiles a
// chunk touches. Measured on the collision's disks in random / in cell order (direct, then tiled,
// us): 98,304 particles on 256 bins 38 / 52, 38 / 40; 196,608 on 512 37 / 47, 43 / 44; 307,200 on
// 640 48 / 46, 54 / 55, 368,640 57 / 60, 52 / 54; 345,600 on 900 52 / 44, 62 / 65, 518,400 82 / 69,
// 72 / 70; 491,520 on 1024 59 / 48, 57 / 58, 589,824 64 / 58, 57 / 59; 10,000,002 on 512 1763 /
// 3447, 133 / 119. So a bin of side wants 384 particles up to 512 bins and 544 above. The launches
// and the passes over short counts cost 18 to 35 us however few the particles, which small images
// reach only with more particles a bin (direct / tiled): 1,000 on 1 bin 19 / 19, 3,000 43 / 28;
// 6,144 on 4 bins 30 / 32, 10,000 44 / 34; 6,144 on 16 bins 23 / 32, 10,000 33 / 34; 40,000 on 100
// 37 / 36. kMaxTiles bounds the bins.
bool use_tiled(int64_t n, int bins) {
  const int64_t least = std::max<int64_t>(int64_t{bins <= 512 ? 384 : 544} * bins,
                                          std::min(2048 * bins, 10240));
  return n >= least && (bins + kTileSide - 1) / kTileSide <= 16;
}

pm_status check_project(const char* who, const float* pos_a, const float* pos_b,
                        const float* mass, int64_t n, float binw_a, float binw_b, int32_t bins,
                        const float* img, const void* scratch) {
  const std::string w(who);
  PM_REQUIRE(img && scratch, w + ": null output or scratch");
  PM_REQUIRE(n >= 0 && n <= (int64_t(1) << 28), w + ": particle count out of range");
  PM_REQUIRE(n == 0 || (pos_a && pos_b && mass), w + ": null particle arrays");
  PM_REQUIRE(bins >= 1 && bins <= 8192, w + ": bins must be in [1, 8192]");
  PM_REQUIRE(binw_a > 0.0f && binw_b > 0.0f, w + ": bin widths must be positive");
  PM_REQUIRE((reinterpret_cast<uintptr_t>(scratch) & 7u) == 0,
             w + ": scratch must be 8-byte aligned");
  return PM_OK;
}

}  // namespace

extern "C" {

pm_status pm_project_mass(const float* pos_a, const float* pos_b, const float* mass, int64_t n,
                          float lo_a, float lo_b, float binw_a, float binw_b, int32_t bins,
                          float* img, void* scratch, hipStream_t s) {
  pm::clear_error();
  pm_status st = check_project("pm_project_mass", pos_a, pos_b, mass, n, binw_a, binw_b, bins,
                               img, scratch);
  if (st) return st;
  const int64_t cells = static_cast<int64_t>(bins) * bins;
  auto* acc = static_cast<unsigned long long*>(scratch);
  auto* maxbits = reinterpret_cast<unsigned int*>(acc + cells);
  PM_TIMED("project", 16.0 * static_cast<double>(n) + 12.0 * static_cast<double>(cells), s);
  // the workgroups' maxima lie in the image until unscale_kernel writes it
  auto* maxima = reinterpret_cast<unsigned int*>(img);
  const int nmax = static_cast<int>(
      std::min({static_cast<int64_t>(pm::stream_blocks(std::max(n, cells + 1))), cells,
                static_cast<int64_t>(kMaxima)}));
  clear_max_kernel<<<static_cast<unsigned>(nmax), 256, 0, s>>>(mass, n, acc, cells, maxima);
  PM_CHECK_LAUNCH("clear_max_kernel");
  if (n > 0) {
    project_kernel<<<pm::stream_blocks(n), 256, 0, s>>>(pos_a, pos_b, mass, n, lo_a, lo_b, binw_a,
                                                        binw_b, bins, maxima, nmax, maxbits, acc);
    PM_CHECK_LAUNCH("project_kernel");
  }
  unscale_kernel<<<pm::blocks_for(cells), 256, 0, s>>>(acc, cells, maxbits, img);
  PM_CHECK_LAUNCH("unscale_kernel");
  return PM_OK;
}

pm_status pm_project_scratch_bytes(int32_t bins, int64_t* out) {
  PM_REQUIRE(out && bins >= 1 && bins <= 8192, "pm_project_scratch_bytes: bad argument");
  *out = (static_cast<int64_t>(bins) * bins + 1) * 8;
  return PM_OK;
}

pm_status pm_project_work_bytes(int64_t n, int32_t bins, int64_t* out) {
  PM_REQUIRE(out && bins >= 1 && bins <= 8192 && n >= 0 && n <= (int64_t(1) << 28),
             "pm_project_work_bytes: bad argument");
  if (!use_tiled(n, bins)) return pm_project_scratch_bytes(bins, out);
  *out = tiled_layout(n, bins).bytes;
  return PM_OK;
}

pm_status pm_project_mass_work(const float* pos_a, const float* pos_b, const float* mass,
                               int64_t n, float lo_a, float lo_b, float binw_a, float binw_b,
                               int32_t bins, float* img, void* work, hipStream_t s) {
  pm::clear_error();
  pm_status st = check_project("pm_project_mass_work", pos_a, pos_b, mass, n, binw_a, binw_b,
                               bins, img, work);
  if (st) return st;
  if (!use_tiled(n, bins))
    return pm_project_mass(pos_a, pos_b, mass, n, lo_a, lo_b, binw_a, binw_b, bins, img, work, s);
  const TiledLayout l = tiled_layout(n, bins);
  char* base = static_cast<char*>(work);
  ProjectArgs a;
  a.pa = pos_a;
  a.pb = pos_b;
  a.mass = mass;
  a.n = n;
  a.lo_a = lo_a;
  a.lo_b = lo_b;
  a.binw_a = binw_a;
  a.binw_b = binw_b;
  a.bins = bins;
  a.tiles_b = l.tiles_b;
  a.tiles = l.tiles;
  a.groups = l.groups;
  a.acc = reinterpret_cast<unsigned long long*>(base + l.acc);
  a.records = reinterpret_cast<unsigned long long*>(base + l.records);
  a.hist = reinterpret_cast<unsigned*>(base + l.hist);
  a.group_max = reinterpret_cast<unsigned*>(base + l.group_max);
  a.totals = reinterpret_cast<unsigned*>(base + l.totals);
  a.maxbits = reinterpret_cast<unsigned*>(base + l.maxbits);
  const int64_t cells = static_cast<int64_t>(bins) * bins;
  PM_TIMED("project", 16.0 * static_cast<double>(n) + 12.0 * static_cast<double>(cells), s);
  tile_count_kernel<<<static_cast<unsigned>(l.groups), 256, 0, s>>>(a);
  PM_CHECK_LAUNCH("tile_count_kernel");
  constexpr int kSlabGroups = static_cast<int>(kSlab / kGroup);
  for (int g0 = 0; g0 < l.groups; g0 += kSlabGroups) {
    const int g1 = std::min(l.groups, g0 + kSlabGroups);
    tile_scan_kernel<<<static_cast<unsigned>(l.tiles), 256, 0, s>>>(a, g0, g1);
    PM_CHECK_LAUNCH("tile_scan_kernel");
    tile_scatter_kernel<<<static_cast<unsigned>(g1 - g0), 256, 0, s>>>(a, g0);
    PM_CHECK_LAUNCH("tile_scatter_kernel");
    const int64_t most = std::min(n, static_cast<int64_t>(g1) * kGroup) -
                         static_cast<int64_t>(g0) * kGroup;
    tile_sum_kernel<<<pm::blocks_for(most, kChunk), 512, 0, s>>>(a);
    PM_CHECK_LAUNCH("tile_sum_kernel");
  }
  unscale_kernel<<<pm::blocks_for(cells), 256, 0, s>>>(a.acc, cells, a.maxbits, img);
  PM_CHECK_LAUNCH("unscale_kernel");
  return PM_OK;
}

}  // extern "C"
