// Device primitives replacing the reference's thrust calls (thrust::sort_by_key and
// thrust::reduce, SPH-3D-2/sph_system.cu:126-128, :1639-1643, :1832-1836):
//   * exclusive scan (deterministic integer reduce-then-scan: per-tile sums, then each tile
//     adds the sums of the tiles before it, which it reads itself when there are at most
//     1024 tiles and otherwise takes from a single-block scan of the sums);
//   * stable LSD radix sort of (cell hash, slot) with digits of up to 9 bits (an 18-bit key,
//     64^3 cells, takes two passes). A pass is two launches: LDS histograms per tile and per
//     group of tiles, and a scatter whose stable in-tile rank comes from 64-lane ballot matching
//     and per-wave digit counts in LDS, and which adds up the groups before its own; above 128
//     groups a third launch between them does that.
// All integer work, no floating point, results independent of scheduling.
#include <mutex>

#include "sph_device.h"

namespace {

constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;  // 2048
constexpr uint SCAN_FUSED_TILES = 4 * SCAN_THREADS;     // two-kernel scan up to 1024 tiles

constexpr int RADIX_BITS = 9;           // widest digit
constexpr int RADIX = 1 << RADIX_BITS;  // 512 bins
constexpr int SORT_ITEMS = 4;        // keys of a thread
constexpr int GROUP_TILES = 4;
constexpr int SORT_TILE_MIN = 256 * SORT_ITEMS;
constexpr uint BASE_GROUPS = 128;    // more groups are added up by a launch of their own

// Waves of a tile for n keys: enough workgroups for the GPU, and few enough groups for a workgroup to
// add up. Beyond 1M keys the groups have their own launch and a tile is 4096 keys, eight of a digit.
inline int sort_waves(size_t n) { return n <= 131072 ? 4 : (n <= 1048576 ? 8 : 16); }

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_reduce(const uint *__restrict__ in,
                                                              const uint *n_dev, uint n_host,
                                                              uint *__restrict__ tmp) {
  __shared__ uint lw[SCAN_THREADS / 64];
  const uint n = n_dev ? min(*n_dev, n_host) : n_host;
  const size_t base = (size_t)blockIdx.x * SCAN_TILE + (size_t)threadIdx.x * SCAN_ITEMS;
  uint s = 0;
#pragma unroll
  for (int j = 0; j < SCAN_ITEMS; j++)
    if (base + j < n) s += in[base + j];
  uint tot;
  block_excl_scan(s, lw, tot);
  if (threadIdx.x == 0) tmp[blockIdx.x] = tot;
}

__global__ __launch_bounds__(1024) void k_scan_top(uint *__restrict__ tmp, const uint *n_dev,
                                                   uint n_host, uint *total_dev) {
  __shared__ uint lw[16];
  const uint n = n_dev ? min(*n_dev, n_host) : n_host;
  const uint nb = (n + SCAN_TILE - 1) / SCAN_TILE;
  uint carry = 0;
  for (uint base = 0; base < nb; base += blockDim.x) {
    uint i = base + threadIdx.x;
    uint v = i < nb ? tmp[i] : 0u;
    uint tot;
    uint ex = block_excl_scan(v, lw, tot);
    if (i < nb) tmp[i] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0 && total_dev) *total_dev = carry;
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_down(const uint *__restrict__ in,
                                                            uint *__restrict__ out,
                                                            const uint *n_dev, uint n_host,
                                                            const uint *__restrict__ tmp) {
  __shared__ uint lw[SCAN_THREADS / 64];
  const uint n = n_dev ? min(*n_dev, n_host) : n_host;
  const size_t base = (size_t)blockIdx.x * SCAN_TILE + (size_t)threadIdx.x * SCAN_ITEMS;
  if ((size_t)blockIdx.x * SCAN_TILE >= n) return;  // uniform per block
  uint v[SCAN_ITEMS];
  uint s = 0;
#pragma unroll
  for (int j = 0; j < SCAN_ITEMS; j++) {
    v[j] = base + j < n ? in[base + j] : 0u;
    s += v[j];
  }
  uint tot;
  uint run = block_excl_scan(s, lw, tot) + tmp[blockIdx.x];
#pragma unroll
  for (int j = 0; j < SCAN_ITEMS; j++) {
    if (base + j < n) out[base + j] = run;
    run += v[j];
  }
}

// Down-sweep that forms its own carry: the sum of the tile sums before this tile (at most
// SCAN_FUSED_TILES of them, up to four per thread, added in a fixed order). The last tile
// writes the total; with n = 0 tile 0 writes a zero total.
__global__ __launch_bounds__(SCAN_THREADS) void k_scan_down_carry(const uint *__restrict__ in,
                                                                  uint *__restrict__ out,
                                                                  const uint *n_dev, uint n_host,
                                                                  const uint *__restrict__ tmp,
                                                                  uint *total_dev) {
  __shared__ uint lw[SCAN_THREADS / 64];
  const uint n = n_dev ? min(*n_dev, n_host) : n_host;
  if (n == 0) {
    if (blockIdx.x == 0 && threadIdx.x == 0 && total_dev) *total_dev = 0u;
    return;
  }
  if ((size_t)blockIdx.x * SCAN_TILE >= n) return;  // uniform per block
  const uint nb = (n + SCAN_TILE - 1) / SCAN_TILE;
  uint part = 0;
  for (uint k = threadIdx.x; k < blockIdx.x; k += SCAN_THREADS) part += tmp[k];
  uint carry;
  block_excl_scan(part, lw, carry);
  const size_t base = (size_t)blockIdx.x * SCAN_TILE + (size_t)threadIdx.x * SCAN_ITEMS;
  uint v[SCAN_ITEMS];
  uint s = 0;
#pragma unroll
  for (int j = 0; j < SCAN_ITEMS; j++) {
    v[j] = base + j < n ? in[base + j] : 0u;
    s += v[j];
  }
  uint tot;
  uint run = block_excl_scan(s, lw, tot) + carry;
#pragma unroll
  for (int j = 0; j < SCAN_ITEMS; j++) {
    if (base + j < n) out[base + j] = run;
    run += v[j];
  }
  if (blockIdx.x == nb - 1 && threadIdx.x == 0 && total_dev) *total_dev = carry + tot;
}

__global__ __launch_bounds__(256) void k_fill(uint *p, uint value, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = value;
}

__global__ __launch_bounds__(256) void k_fill2(uint *a, uint va, uint *b, uint vb, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    a[i] = va;
    b[i] = vb;
  }
}

// Keys to sort: the device count when given (clamped to the host bound), else the host's.
__device__ inline uint sort_count(const uint *n_dev, uint n_host) {
  return n_dev ? min(*n_dev, n_host) : n_host;
}

// Bins of a digit: whole 16-byte groups (the first pass over one bit has two that stay empty).
__device__ __host__ inline uint radix_bins(int width) { return width < 2 ? 4u : 1u << width; }

// Histograms of a pass: workgroup b takes groups b, b + gridDim.x, ... of GROUP_TILES tiles.
// pre[tile * bins + d]: keys of digit d in the group's tiles before this one; gsum[group *
// bins + d]: in the whole group.
template <int W>
__global__ __launch_bounds__(64 * W) void k_radix_hist(const uint *__restrict__ keys,
                                                             const uint *n_dev, uint n_host,
                                                             int shift, int width,
                                                             uint *__restrict__ pre,
                                                             uint *__restrict__ gsum) {
  constexpr uint SORT_THREADS = 64 * W, SORT_TILE = SORT_THREADS * SORT_ITEMS;
  constexpr int PER_WAVE = GROUP_TILES * SORT_TILE / W;  // keys of a wave
  constexpr int TILE_WAVES = W / GROUP_TILES;
  __shared__ uint h[GROUP_TILES][RADIX];
  const uint t = threadIdx.x, lane = t & 63u, w = t >> 6;
  const uint nbin = radix_bins(width), mask = (1u << width) - 1u;
  const uint n = sort_count(n_dev, n_host);
  const uint ntiles = (n + SORT_TILE - 1) / SORT_TILE;
  const uint ngroups = (ntiles + GROUP_TILES - 1) / GROUP_TILES;
  for (uint g = blockIdx.x; g < ngroups; g += gridDim.x) {
    for (uint x = t; x < GROUP_TILES * RADIX; x += SORT_THREADS) (&h[0][0])[x] = 0u;
    __syncthreads();
    const size_t base = (size_t)g * GROUP_TILES * SORT_TILE + w * PER_WAVE + lane;
    uint *const hw = h[w / TILE_WAVES];
#pragma unroll
    for (int j = 0; j < PER_WAVE / 64; j++) {
      const size_t i = base + 64 * j;
      if (i < n) atomicAdd(&hw[(keys[i] >> shift) & mask], 1u);
    }
    __syncthreads();
    for (uint d = t; d < nbin; d += SORT_THREADS) {
      uint a = 0;
#pragma unroll
      for (int k = 0; k < GROUP_TILES; k++) {
        const uint tile = g * GROUP_TILES + k;
        if (tile < ntiles) pre[(size_t)tile * nbin + d] = a;
        a += h[k][d];
      }
      gsum[(size_t)g * nbin + d] = a;
    }
    __syncthreads();  // h is cleared for the next group
  }
}

// gsum[group][d] becomes the sum over the groups before, total[d] the sum over all. A workgroup
// takes BASE_DIGITS digits; a thread sums a run of groups, the runs are scanned in LDS.
constexpr int BASE_THREADS = 1024, BASE_DIGITS = 32, BASE_ROWS = BASE_THREADS / BASE_DIGITS;
__global__ __launch_bounds__(BASE_THREADS) void k_radix_base(const uint *n_dev, uint n_host, int width,
                                                             uint group_keys,
                                                             uint *__restrict__ gsum,
                                                             uint *__restrict__ total) {
  __shared__ uint s[BASE_ROWS][BASE_DIGITS];
  const uint nbin = radix_bins(width);
  const uint n = sort_count(n_dev, n_host);
  const uint ngroups = (n + group_keys - 1) / group_keys;
  const uint x = threadIdx.x % BASE_DIGITS, r = threadIdx.x / BASE_DIGITS;
  const uint d = blockIdx.x * BASE_DIGITS + x;
  const uint len = (ngroups + BASE_ROWS - 1) / BASE_ROWS, g0 = min(r * len, ngroups), g1 = min(g0 + len, ngroups);
  uint sum = 0;
  if (d < nbin)
    for (uint g = g0; g < g1; g++) sum += gsum[(size_t)g * nbin + d];
  s[r][x] = sum;
  __syncthreads();
  uint run = 0, all = 0;
  for (uint k = 0; k < BASE_ROWS; k++) {
    run += k < r ? s[k][x] : 0u;
    all += s[k][x];
  }
  if (d >= nbin) return;
  for (uint g = g0; g < g1; g++) {
    const uint v = gsum[(size_t)g * nbin + d];
    gsum[(size_t)g * nbin + d] = run;
    run += v;
  }
  if (r == 0) total[d] = all;
}

// Stable scatter. A wave takes SORT_ITEMS rounds of 64 consecutive keys and counts its digits in
// its own row of LDS, so no round needs a block barrier: the rank of a key among equal digits is
// the row's count from earlier rounds plus the equal digits in lower lanes (ballot match). Then
// each digit's row counts become places: the smaller digits of all keys, this digit's of the
// groups before (both from k_radix_base, or added up here when total is null), of the group's
// tiles before and of the tile's waves before. The tile is put in order in LDS first, so that its
// stores go out in runs of a digit (700k keys, a digit of 9 bits: 22.6 -> 17.5 us). Bound: the
// scattered stores and, up to some 100k keys, the chain of loads. Against a digit-major histogram,
// its scan in two launches and a scatter with three barriers per round, us per call of
// sph_sort_noalloc: 700k keys of 27 bits 110 -> 77, 1M 145 -> 91, 100k 60 -> 56, 1000 40 -> 35;
// 700k of 18 bits 71 -> 49, of 32 bits 110 -> 80.
template <int W>
__global__ __launch_bounds__(64 * W) void k_radix_scatter(
    const uint *__restrict__ keys_in, const uint *__restrict__ vals_in, const uint *n_dev,
    uint n_host, int shift, int width, const uint *__restrict__ pre, const uint *__restrict__ gsum,
    const uint *__restrict__ total, uint *__restrict__ keys_out, uint *__restrict__ vals_out) {
  constexpr uint SORT_THREADS = 64 * W, SORT_TILE = SORT_THREADS * SORT_ITEMS;
  constexpr uint DP = RADIX > SORT_THREADS ? RADIX / SORT_THREADS : 1;  // a thread's digits
  __shared__ uint cnt[W][RADIX];
  __shared__ uint all[RADIX], before[RADIX];
  __shared__ uint skey[SORT_TILE], sval[SORT_TILE];
  __shared__ uint lw[W];
  const uint t = threadIdx.x, lane = t & 63u, w = t >> 6;
  const uint nbin = radix_bins(width), mask = (1u << width) - 1u;
  const uint n = sort_count(n_dev, n_host);
  const uint ntiles = (n + SORT_TILE - 1) / SORT_TILE;
  const uint ngroups = (ntiles + GROUP_TILES - 1) / GROUP_TILES;
  const unsigned long long lt = (1ull << lane) - 1ull;
  for (uint tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const uint g = tile / GROUP_TILES;
    const size_t base = (size_t)tile * SORT_TILE + w * (64 * SORT_ITEMS) + lane;
    uint key[SORT_ITEMS], val[SORT_ITEMS], rank[SORT_ITEMS], mine[DP];
#pragma unroll
    for (int j = 0; j < SORT_ITEMS; j++) {
      const size_t i = base + 64 * j;
      key[j] = i < n ? keys_in[i] : 0u;
      val[j] = i < n ? (vals_in ? vals_in[i] : (uint)i) : 0u;
    }
#pragma unroll
    for (uint k = 0; k < DP; k++) mine[k] = t * DP + k < nbin ? pre[(size_t)tile * nbin + t * DP + k] : 0u;
    for (uint x = t; x < W * RADIX; x += SORT_THREADS) (&cnt[0][0])[x] = 0u;
    for (uint x = t; x < RADIX; x += SORT_THREADS) all[x] = before[x] = 0u;
    __syncthreads();
    if (total) {
      for (uint d = t; d < nbin; d += SORT_THREADS) {
        all[d] = total[d];
        before[d] = gsum[(size_t)g * nbin + d];
      }
    } else {  // four digits of every few groups
      const uint quads = nbin / 4u, q = t & (quads - 1u), rows = SORT_THREADS / quads;
      uint4 a = make_uint4(0u, 0u, 0u, 0u), b = a;
#pragma unroll 8
      for (uint r = t / quads; r < ngroups; r += rows) {
        const uint4 v = reinterpret_cast<const uint4 *>(gsum)[(size_t)r * quads + q];
        const uint m = r < g ? 0xffffffffu : 0u;
        a = make_uint4(a.x + v.x, a.y + v.y, a.z + v.z, a.w + v.w);
        b = make_uint4(b.x + (v.x & m), b.y + (v.y & m), b.z + (v.z & m), b.w + (v.w & m));
      }
      atomicAdd(&all[4 * q], a.x), atomicAdd(&all[4 * q + 1], a.y);
      atomicAdd(&all[4 * q + 2], a.z), atomicAdd(&all[4 * q + 3], a.w);
      atomicAdd(&before[4 * q], b.x), atomicAdd(&before[4 * q + 1], b.y);
      atomicAdd(&before[4 * q + 2], b.z), atomicAdd(&before[4 * q + 3], b.w);
    }
#pragma unroll
    for (int j = 0; j < SORT_ITEMS; j++) {
      const bool valid = base + 64 * j < n;
      const uint d = (key[j] >> shift) & mask;
      unsigned long long peers = __ballot(valid);
      for (int b = 0; b < width; b++) {  // width is uniform: the ballots stay wave-wide
        const unsigned long long bb = __ballot((d >> b) & 1u);
        peers &= ((d >> b) & 1u) ? bb : ~bb;
      }
      const uint lower = (uint)__popcll(peers & lt);
      const uint seen = cnt[w][d];
      rank[j] = seen + lower;
      // the row is read by every lane before its digits' first lanes write it, and written
      // before the next round reads it
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (valid && lower == 0u) cnt[w][d] = seen + (uint)__popcll(peers);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    uint tot, sum = 0, here = 0, local[DP];
#pragma unroll
    for (uint k = 0; k < DP; k++) {
      const uint d = t * DP + k;
      local[k] = 0u;
      if (d < nbin) {
        sum += all[d];
#pragma unroll
        for (int x = 0; x < W; x++) local[k] += cnt[x][d];
        here += local[k];
      }
    }
    uint smaller = block_excl_scan(sum, lw, tot);  // keys of smaller digits: in all
    uint at = block_excl_scan(here, lw, tot);      // and in this tile
#pragma unroll
    for (uint k = 0; k < DP; k++) {
      const uint d = t * DP + k;
      if (d < nbin) {
        before[d] = smaller + before[d] + mine[k] - at;  // place of a key - its place in the tile
        uint q = at;
#pragma unroll
        for (int x = 0; x < W; x++) {
          const uint c = cnt[x][d];
          cnt[x][d] = q;
          q += c;
        }
        smaller += all[d];
        at += local[k];
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < SORT_ITEMS; j++)
      if (base + 64 * j < n) {
        const uint q = cnt[w][(key[j] >> shift) & mask] + rank[j];
        skey[q] = key[j];
        sval[q] = val[j];
      }
    __syncthreads();
#pragma unroll
    for (uint j = 0; j < SORT_ITEMS; j++) {  // a digit's keys side by side
      const uint q = j * SORT_THREADS + t;
      if (q < tot) {
        const uint k = skey[q], to = before[(k >> shift) & mask] + q;
        keys_out[to] = k;
        vals_out[to] = sval[q];
      }
    }
    __syncthreads();  // the counts start over
  }
}

inline uint blocks_for(size_t n, size_t per) { return (uint)((n + per - 1) / per); }

}  // namespace

size_t sph_scan_tmp_elems(size_t n) { return (n + SCAN_TILE - 1) / SCAN_TILE + 1; }
// per tile, per group and one row of totals, for any tile size
size_t sph_sort_hist_elems(size_t n) {
  const size_t tiles = (n + SORT_TILE_MIN - 1) / SORT_TILE_MIN;
  return (size_t)RADIX * (tiles + (tiles + GROUP_TILES - 1) / GROUP_TILES + 1);
}

void sph_exclusive_scan(const uint *in, uint *out, const uint *n_dev, uint n_max, uint *total_dev,
                        uint *tmp, hipStream_t st) {
  uint nb = blocks_for(n_max, SCAN_TILE);
  if (nb == 0) nb = 1;
  if (nb <= SCAN_FUSED_TILES) {
    hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(SCAN_THREADS), 0, st, in, n_dev, n_max, tmp);
    hipLaunchKernelGGL(k_scan_down_carry, dim3(nb), dim3(SCAN_THREADS), 0, st, in, out, n_dev,
                       n_max, tmp, total_dev);
    return;
  }
  hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(SCAN_THREADS), 0, st, in, n_dev, n_max, tmp);
  hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, st, tmp, n_dev, n_max, total_dev);
  hipLaunchKernelGGL(k_scan_down, dim3(nb), dim3(SCAN_THREADS), 0, st, in, out, n_dev, n_max, tmp);
}

void sph_fill_u32(uint *p, uint value, size_t n, hipStream_t st) {
  if (n == 0) return;
  size_t nb = (n + 255) / 256;
  if (nb > 65536) nb = 65536;
  hipLaunchKernelGGL(k_fill, dim3((uint)nb), dim3(256), 0, st, p, value, n);
}

// Undo launch_cell_bounds over the same sorted keys: the cells at the run starts get their
// fill values back (the other cells were never written).
__global__ __launch_bounds__(256) void k_reset_cells(const uint *__restrict__ skeys, uint n,
                                                     uint ncell, uint *__restrict__ cstart,
                                                     uint *__restrict__ cend) {
  const uint k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  const uint h = skeys[k];
  if (h < ncell && (k == 0 || skeys[k - 1] != h)) {
    cstart[h] = SPH_EMPTY;
    cend[h] = 0u;
  }
}

void sph_reset_cells(const uint *skeys, uint n, uint ncell, uint *cstart, uint *cend,
                     hipStream_t st) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_reset_cells, dim3((n + 255) / 256), dim3(256), 0, st, skeys, n, ncell,
                     cstart, cend);
}

void sph_fill_cells(uint *cstart, uint *cend, size_t n, hipStream_t st) {
  if (n == 0) return;
  size_t nb = (n + 255) / 256;
  if (nb > 65536) nb = 65536;
  hipLaunchKernelGGL(k_fill2, dim3((uint)nb), dim3(256), 0, st, cstart, SPH_EMPTY, cend, 0u, n);
}

namespace {

// LSD passes over keys[0..n): pass 0 reads (k0, v0) -- v0 == nullptr: the values are the
// indices 0..n-1 -- and writes (k1, v1); each later pass reads what the one before wrote
// and writes the other pair, (vbuf0 standing in as v0's storage). The result ends in
// (*keys_out, *vals_out).
// n_dev (optional): a device word holding the key count, n only bounding it; grid
// (optional): a persistent grid for the histogram and scatter kernels.
void radix_passes(uint *k0, const uint *v0, uint *vbuf0, uint *k1, uint *v1, uint n, int bits,
                  uint *tile_hist, uint **keys_out, uint **vals_out, hipStream_t st,
                  const uint *n_dev = nullptr, uint grid = 0) {
  const uint *kin = k0, *vin = v0;
  uint *kout = k1, *vout = v1;
  const int waves = sort_waves(n);
  const uint threads = 64u * waves, tile_keys = threads * SORT_ITEMS;
  const uint ntiles = blocks_for(n, tile_keys), ngroups = blocks_for(ntiles, GROUP_TILES);
  const bool based = ngroups > BASE_GROUPS;
  if (bits < 1) bits = 1;
  // fewest passes of at most RADIX_BITS bits, the digit width spread evenly over them
  const int passes = (bits + RADIX_BITS - 1) / RADIX_BITS;
  const int width = (bits + passes - 1) / passes;
  uint *const gsum = tile_hist + (size_t)RADIX * ntiles, *const total = gsum + (size_t)RADIX * ngroups;
  for (int p = 0; p < passes && n > 0; p++) {
    const int shift = p * width;
#define SPH_RADIX(KERNEL, blocks, ...)                                                       \
  do {                                                                                       \
    const dim3 g(grid ? grid : (blocks)), b(threads);                                        \
    if (waves == 4) KERNEL<4><<<g, b, 0, st>>>(__VA_ARGS__);                                  \
    else if (waves == 8) KERNEL<8><<<g, b, 0, st>>>(__VA_ARGS__);                             \
    else KERNEL<16><<<g, b, 0, st>>>(__VA_ARGS__);                                            \
  } while (0)
    SPH_RADIX(k_radix_hist, ngroups, kin, n_dev, n, shift, width, tile_hist, gsum);
    if (based)
      hipLaunchKernelGGL(k_radix_base, dim3(blocks_for(radix_bins(width), BASE_DIGITS)), dim3(BASE_THREADS),
                         0, st, n_dev, n, width, GROUP_TILES * tile_keys, gsum, total);
    SPH_RADIX(k_radix_scatter, ntiles, kin, vin, n_dev, n, shift, width, tile_hist, gsum,
              based ? total : nullptr, kout, vout);
#undef SPH_RADIX
    // next pass reads what this one wrote
    uint *nk = kout, *nv = vout;
    if (kout == k1) {
      kout = k0;
      vout = vbuf0;
    } else {
      kout = k1;
      vout = v1;
    }
    kin = nk;
    vin = nv;
  }
  *keys_out = const_cast<uint *>(kin);
  *vals_out = const_cast<uint *>(vin);
}

}  // namespace

void sph_radix_sort(uint *keys, uint *vals, uint n, int bits, SortScratch &sc, uint **keys_out,
                    uint **vals_out, hipStream_t st, const uint *n_dev, uint grid) {
  radix_passes(keys, nullptr, vals, sc.keys_alt, sc.vals_alt, n, bits, sc.tile_hist, keys_out,
               vals_out, st, n_dev, grid);
}

// ---------------------------------------------------------------------------------------
// Sort without allocation. The sort's working memory (ping-pong partners, histograms) is one static device array instead of buffers a context allocates, so
// the call makes no hipMalloc/hipFree: for callers that cannot allocate (code under stream
// capture into a graph, serving loops that forbid allocation). Each GPU holds its own copy
// of the array for the life of the process; every call on one GPU shares it, so calls that
// overlap on one GPU (other streams, other threads) race. Nothing in it needs clearing:
// every pass writes the histogram entries it scans before reading them.
// ---------------------------------------------------------------------------------------
namespace {
constexpr uint kNoAllocMaxKeys = 1u << 20;
constexpr size_t kNoAllocTiles = (kNoAllocMaxKeys + SORT_TILE_MIN - 1) / SORT_TILE_MIN;
constexpr size_t kNoAllocHist = (size_t)RADIX * (kNoAllocTiles + (kNoAllocTiles + GROUP_TILES - 1) / GROUP_TILES + 1);
// [keys_alt | vals_alt | histograms], every part 256-byte aligned
constexpr size_t kNoAllocKeysAlt = 0;
constexpr size_t kNoAllocValsAlt = kNoAllocKeysAlt + kNoAllocMaxKeys;
constexpr size_t kNoAllocHistOff = kNoAllocValsAlt + kNoAllocMaxKeys;
constexpr size_t kNoAllocWords = kNoAllocHistOff + kNoAllocHist;
static_assert(kNoAllocHistOff % 64 == 0, "scratch part alignment");
static_assert(SPH_SORT_NOALLOC_MAX_KEYS == kNoAllocMaxKeys, "header limit");
}  // namespace

static __device__ __align__(256) uint scratch[kNoAllocWords];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
uint *g_scratch_dev[kMaxDevices] = {};  // device address of `scratch`, per GPU

// The device address of this GPU's copy of `scratch`, looked up once per device (with that
// device current) on its first call. The array's host-side name is not a device address.
int noalloc_scratch(uint **out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) return SPH_EHIP;
  if (dev < 0 || dev >= kMaxDevices) return SPH_EINVAL;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return SPH_EHIP;
    g_scratch_dev[dev] = (uint *)p;
  }
  *out = g_scratch_dev[dev];
  return SPH_OK;
}

__global__ __launch_bounds__(256) void k_copy_pairs(const uint *__restrict__ ka,
                                                    const uint *__restrict__ va, uint *__restrict__ kb,
                                                    uint *__restrict__ vb, uint n) {
  const uint i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) {
    kb[i] = ka[i];
    vb[i] = va[i];
  }
}
}  // namespace

extern "C" int sph_sort_noalloc(uint32_t *hash, uint32_t *index, uint32_t n, uint32_t key_bits,
                                void *stream) {
  if (n == 0) return SPH_OK;
  if (!hash || !index || key_bits > 32) return SPH_EINVAL;
  if (n > kNoAllocMaxKeys) return SPH_ECAP;
  uint *base = nullptr;
  int rc = noalloc_scratch(&base);
  if (rc != SPH_OK) return rc;
  hipStream_t st = (hipStream_t)stream;
  uint *ko = nullptr, *vo = nullptr;
  radix_passes(hash, index, index, base + kNoAllocKeysAlt, base + kNoAllocValsAlt, n,
               key_bits ? (int)key_bits : 32, base + kNoAllocHistOff, &ko, &vo, st);
  if (ko != hash)  // an odd number of passes ends in the scratch pair
    hipLaunchKernelGGL(k_copy_pairs, dim3((n + 255) / 256), dim3(256), 0, st, ko, vo, hash, index, n);
  return hipGetLastError() == hipSuccess ? SPH_OK : SPH_EHIP;
}

// A plain copy of n 16-byte units: one load and one store per unit, grid-stride.
__global__ __launch_bounds__(256) void k_copy_calibration(const float4 *__restrict__ src,
                                                          float4 *__restrict__ dst, size_t n) {
  const size_t stride = (size_t)gridDim.x * 256;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

extern "C" int sph_copy_calibration(size_t bytes, int reps) {
  const size_t n = bytes / 16;
  if (n == 0 || reps <= 0) return SPH_EINVAL;
  float4 *src = nullptr, *dst = nullptr;
  if (hipMalloc(&src, n * 16) != hipSuccess) return SPH_ECAP;
  if (hipMalloc(&dst, n * 16) != hipSuccess) {
    (void)hipFree(src);
    return SPH_ECAP;
  }
  hipError_t e = hipMemset(src, 0, n * 16);
  const size_t blocks = std::min<size_t>((n + 255) / 256, 256 * 32);
  for (int r = 0; r < reps && e == hipSuccess; r++) {
    k_copy_calibration<<<dim3((uint)blocks), dim3(256), 0, 0>>>(src, dst, n);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipDeviceSynchronize();
  (void)hipFree(src);
  (void)hipFree(dst);
  return e == hipSuccess ? SPH_OK : SPH_EHIP;
}
