// Cell order without a sort by key (A1-A4 of the step, SPH-3D-2/sph_system.cu:78-202): the
// particles are counted into their cells, the counts are scanned into the cell table, and
// each particle finds its place in its cell by counting the smaller slots there. The result is
// the order of the stable sort of (cell hash, slot), the cell table and the reordered state, in
// four or five launches instead of the thirteen of hash, radix sort (two digit passes), table
// fill, run boundaries and gather:
//   k_bin_count    cell of each entry; its arrival rank in the cell from an atomic counter
//   k_bin_scan     one block over up to SCAN1_CELLS cells; more cells take two launches,
//                  tile sums (k_bin_tiles) and a scan that adds the sums before its tile
//   k_bin_place    each entry's slot into its cell's stretch, in arrival order
//   k_bin_reorder  an entry's place = cell start + entries of the cell with a smaller slot; the
//                  record goes there
// The arrival order differs from run to run, the places do not. Bound: launches and latency up
// to some 100k particles, HBM beyond (the records move once: 52 bytes read, 64 written).
// Counting needs a scan over all cells, so a sparse grid keeps the radix sort (sph_use_bins); so
// does the step after one that found particles outside the grid, which share a cell however many
// they are (k_bin_reorder reads a cell once per entry).
#include <algorithm>

#include "sph_device.h"

namespace {

constexpr int CS_ITEMS = 8;                 // cells per thread of a scan
constexpr uint CS_TILE = BLK * CS_ITEMS;    // 2048 cells per block
constexpr uint SCAN1_THREADS = 1024, SCAN1_TILE = SCAN1_THREADS * CS_ITEMS;
constexpr uint SCAN1_CELLS = SCAN1_TILE;  // a second round costs more than a second launch (7.2 us at 13,824)

// A block's entries are counted in LDS first, in a hash table of their cells, so the cell
// counters see one atomic per block and cell instead of one per entry: consecutive entries were
// neighbours a step ago. Atomics that return a value ran at 12.5 G/s whatever the order of the
// blocks: 498k particles 38.7 -> 17.7 us, 3.2M in a batch 75 -> 48 us, 14k 4.9 -> 4.6 us. Four
// entries per thread (a table of 2048 places) were slower, 22.6 and 62 us.
constexpr uint CT = 2 * BLK;  // table places; at most BLK are taken, so every search ends
static_assert(CT == 512, "k_bin_count's hash gives 9 bits");

template <int V, bool B>
__global__ __launch_bounds__(BLK) void k_bin_count(DevParams P0, const DevParams *__restrict__ Ptab,
                                                   SceneCnt *scn, const float4 *__restrict__ pos,
                                                   const uint *__restrict__ slot, uint m_host,
                                                   uint *__restrict__ hkey, uint *__restrict__ rank,
                                                   uint *__restrict__ ccount, Counters *cnt, int par) {
  __shared__ uint tcell[CT], tcnt[CT];
  const uint t = threadIdx.x;
  if (blockIdx.x == 0 && t == 0) {
    cnt->m_in = cnt->m;  // the entries of this step: m itself changes in k_bin_reorder
    if (!B) {            // the step's counters start over (no thread here reads them)
      cnt->n_pre = cnt->n;
      cnt->s_req = cnt->s_done = cnt->groups = 0u;
      cnt->err2[par ^ 1] = 0u;
    }
  }
  const uint m = min(cnt->m, m_host), nvb = (m + BLK - 1) / BLK;
  for (uint vb = blockIdx.x; vb < nvb; vb += gridDim.x) {
    const uint k = vb * BLK + t;
    const uint w = k < m ? slot[k] : SPH_DEAD;
    const bool live = w != SPH_DEAD;
    tcell[t] = tcell[t + BLK] = SPH_EMPTY;
    tcnt[t] = tcnt[t + BLK] = 0u;
    uint h = 0u, at = 0u, r = 0u;
    if (live) {
      const DevParams &P = scene_params<B>(P0, Ptab, w);
      const float4 p = pos[k];
      uint c[3];
      h = P.cell_base;
      if (cell_of<V>(P, p.x, p.y, p.z, c)) {
        h += c[2] * P.ncell[0] * P.ncell[1] + c[1] * P.ncell[0] + c[0];
      } else {  // the scene's cell 0 keeps every later access in bounds
        if (B) {
          atomicOr(&cnt->err, 1u);
          atomicOr(&scn[w >> SPH_SCENE_SHIFT].err, 1u);
        } else {
          atomicOr(&cnt->err2[par], 1u);
        }
      }
      hkey[k] = h;
    }
    __syncthreads();
    if (live) {
      at = (h * 0x9e3779b1u) >> 23;  // the top 9 bits: CT places
      for (;; at = (at + 1u) % CT) {
        const uint was = atomicCAS(&tcell[at], SPH_EMPTY, h);
        if (was == SPH_EMPTY || was == h) break;
      }
      r = atomicAdd(&tcnt[at], 1u);
    }
    __syncthreads();
    for (uint x = t; x < CT; x += BLK)
      if (tcnt[x]) tcnt[x] = atomicAdd(&ccount[tcell[x]], tcnt[x]);
    __syncthreads();
    if (live) rank[k] = tcnt[at] + r;
    __syncthreads();  // the table starts over
  }
}

// counts [c, c + 8) of the table, cleared for the next step; 0 past its end
__device__ inline void take_counts(uint *__restrict__ ccount, size_t c, uint ncell, bool clear,
                                   uint v[CS_ITEMS]) {
  if (c + CS_ITEMS <= ncell) {
    uint4 *const q = reinterpret_cast<uint4 *>(ccount + c);
    const uint4 a = q[0], b = q[1];
    if (clear) q[0] = q[1] = make_uint4(0u, 0u, 0u, 0u);
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
    v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
  } else {
#pragma unroll
    for (int k = 0; k < CS_ITEMS; k++) {
      v[k] = c + k < ncell ? ccount[c + k] : 0u;
      if (clear && c + k < ncell) ccount[c + k] = 0u;
    }
  }
}

// table entries of cells [c, c + 8) from their counts and the particles before them
__device__ inline void put_ranges(uint *__restrict__ cstart, uint *__restrict__ cend, size_t c,
                                  uint ncell, uint run, const uint v[CS_ITEMS]) {
  uint s[CS_ITEMS], e[CS_ITEMS];
#pragma unroll
  for (int k = 0; k < CS_ITEMS; k++) {
    s[k] = v[k] ? run : SPH_EMPTY;
    run += v[k];
    e[k] = v[k] ? run : 0u;
  }
  if (c + CS_ITEMS <= ncell) {
    uint4 *const a = reinterpret_cast<uint4 *>(cstart + c), *const b = reinterpret_cast<uint4 *>(cend + c);
    a[0] = make_uint4(s[0], s[1], s[2], s[3]);
    a[1] = make_uint4(s[4], s[5], s[6], s[7]);
    b[0] = make_uint4(e[0], e[1], e[2], e[3]);
    b[1] = make_uint4(e[4], e[5], e[6], e[7]);
  } else {
#pragma unroll
    for (int k = 0; k < CS_ITEMS; k++)
      if (c + k < ncell) {
        cstart[c + k] = s[k];
        cend[c + k] = e[k];
      }
  }
}

// a single scene's domain errors of this step (collected apart, so that the counting kernel
// could clear the next step's word) become the step's; `keep` adds to what is there
__device__ inline void publish_err(Counters *cnt, int par, bool keep) {
  const uint e = cnt->err2[par];
  cnt->err = keep ? cnt->err | e : e;
}

__global__ __launch_bounds__(SCAN1_THREADS) void k_bin_scan(uint *__restrict__ ccount, uint ncell,
                                                            uint *__restrict__ cstart,
                                                            uint *__restrict__ cend, Counters *cnt,
                                                            int par, bool single, bool keep) {
  __shared__ uint lw[SCAN1_THREADS / 64];
  if (single && threadIdx.x == 0) publish_err(cnt, par, keep);
  const size_t c = (size_t)threadIdx.x * CS_ITEMS;
  uint v[CS_ITEMS], s = 0, tot;
  take_counts(ccount, c, ncell, true, v);
#pragma unroll
  for (int k = 0; k < CS_ITEMS; k++) s += v[k];
  const uint ex = block_excl_scan(s, lw, tot);
  put_ranges(cstart, cend, c, ncell, ex, v);
}

__global__ __launch_bounds__(BLK) void k_bin_tiles(uint *__restrict__ ccount, uint ncell,
                                                   uint *__restrict__ tmp) {
  __shared__ uint lw[BLK / 64];
  uint v[CS_ITEMS], s = 0, tot;
  take_counts(ccount, (size_t)blockIdx.x * CS_TILE + (size_t)threadIdx.x * CS_ITEMS, ncell, false, v);
#pragma unroll
  for (int k = 0; k < CS_ITEMS; k++) s += v[k];
  block_excl_scan(s, lw, tot);
  if (threadIdx.x == 0) tmp[blockIdx.x] = tot;
}

// Each block adds the tile sums before its own itself: at 2048 cells per tile that is one sum
// per 8 kB of table, read from L2.
__global__ __launch_bounds__(BLK) void k_bin_ranges(uint *__restrict__ ccount, uint ncell,
                                                    const uint *__restrict__ tmp,
                                                    uint *__restrict__ cstart, uint *__restrict__ cend,
                                                    Counters *cnt, int par, bool single, bool keep) {
  __shared__ uint lw[BLK / 64];
  if (single && blockIdx.x == 0 && threadIdx.x == 0) publish_err(cnt, par, keep);
  uint part = 0, carry, tot;
  for (uint k = threadIdx.x; k < blockIdx.x; k += BLK) part += tmp[k];
  const size_t c = (size_t)blockIdx.x * CS_TILE + (size_t)threadIdx.x * CS_ITEMS;
  uint v[CS_ITEMS], s = 0;
  take_counts(ccount, c, ncell, true, v);
#pragma unroll
  for (int k = 0; k < CS_ITEMS; k++) s += v[k];
  block_excl_scan(part, lw, carry);
  const uint ex = block_excl_scan(s, lw, tot);
  put_ranges(cstart, cend, c, ncell, carry + ex, v);
}

// zero0, zero1 (optional): the bit arrays that the step's split and merge set, cleared for the
// particles (zero0) and for them and their children (zero1), at most zmax words.
__global__ __launch_bounds__(BLK) void k_bin_place(const uint *__restrict__ slot,
                                                   const uint *__restrict__ hkey,
                                                   const uint *__restrict__ rank,
                                                   const uint *__restrict__ cstart,
                                                   const Counters *cnt, uint m_host,
                                                   uint *__restrict__ bslot, uint *__restrict__ zero0,
                                                   uint *__restrict__ zero1, uint per_split, uint zmax) {
  const uint m = min(cnt->m_in, m_host), z = (m + 31u) / 32u, z1 = min(z * (1u + per_split), zmax);
  for (uint x = blockIdx.x * BLK + threadIdx.x; x < z1; x += gridDim.x * BLK) {
    if (zero0 && x < z) zero0[x] = 0u;
    if (zero1) zero1[x] = 0u;
  }
  for_each_item<false>(m, [&](const uint k) {
    const uint w = slot[k];
    if (w != SPH_DEAD) bslot[cstart[hkey[k]] + rank[k]] = w;
  });
}

// all == false leaves out acc, dp and energy, which the step's force, density and energy
// kernels overwrite for every particle before anything reads them. init (optional, two
// arrays): entry p of both becomes SPH_DEAD.
template <bool B>
__global__ __launch_bounds__(BLK) void k_bin_reorder(DevState src, DevState dst,
                                                     const SceneCnt *__restrict__ scn,
                                                     const uint *__restrict__ hkey,
                                                     const uint *__restrict__ cstart,
                                                     const uint *__restrict__ cend,
                                                     const uint *__restrict__ bslot, Counters *cnt,
                                                     uint m_host, uint *__restrict__ skeys,
                                                     uint *__restrict__ svals, uint *__restrict__ s2p,
                                                     bool all, bool set_m, uint *__restrict__ init0,
                                                     uint *__restrict__ init1, QPosOut qo) {
  if (set_m && blockIdx.x == 0 && threadIdx.x == 0) cnt->m = cnt->n;  // physical == live
  // XCD-contiguous blocks keep a single scene's destinations in one L2 (498k: 24.4 -> 22 us); a
  // batch's were slower that way (81 -> 96 us)
  for_each_item<!B>(min(cnt->m_in, m_host), [&](const uint k) {
    const uint w = src.slot[k];
    if (w == SPH_DEAD) return;
    const float4 p = src.pos[k], v = src.vel[k], e = src.ev[k];
    const uint h = hkey[k], s = cstart[h], t = cend[h];
    uint q = s;
    for (uint j = s; j < t; j += 4) {  // four loads in flight; past the end: the last again
      const uint l = t - 1u;
      const uint a = bslot[j], b = bslot[min(j + 1u, l)], c = bslot[min(j + 2u, l)],
                 d = bslot[min(j + 3u, l)];
      q += (uint)(a < w) + (uint)((b < w) & (j + 1u < t)) + (uint)((c < w) & (j + 2u < t)) +
           (uint)((d < w) & (j + 3u < t));
    }
    dst.pos[q] = p;
    put_qpos<B>(qo, q, w, p);
    dst.vel[q] = v;
    dst.ev[q] = e;
    if (all) {
      dst.acc[q] = src.acc[k];
      dst.dp[q] = src.dp[k];
      dst.energy[q] = src.energy[k];
    }
    dst.slot[q] = w;
    skeys[q] = h;
    const uint d = B ? scn[w >> SPH_SCENE_SHIFT].first + (w & SPH_LOCAL_MASK) : w;
    svals[q] = d;
    s2p[d] = q;
    if (init0) init0[q] = SPH_DEAD;
    if (init1) init1[q] = SPH_DEAD;
  });
}

inline dim3 bgrid(uint grid, size_t n) { return dim3(grid ? grid : (uint)((n + BLK - 1) / BLK)); }

}  // namespace

bool sph_use_bins(size_t total_cell, size_t n) {
  return total_cell <= ((size_t)1 << 22) || total_cell <= 8 * n;
}
size_t sph_bin_tiles(size_t total_cell) { return (total_cell + CS_TILE - 1) / CS_TILE; }

void launch_bin_count(int variant, const DevParams &P, DevState src, const BinScratch &bs,
                      Counters *cnt, uint m, int par, hipStream_t st, const BatchView *bv, uint grid) {
  if (m == 0) return;
#define SPH_BIN_COUNT(V, B)                                                                      \
  k_bin_count<V, B><<<bgrid(grid, m), dim3(BLK), 0, st>>>(P, bv ? bv->Ptab : nullptr,            \
                                                          bv ? bv->scn : nullptr, src.pos, src.slot, \
                                                          m, bs.hkey, bs.rank, bs.ccount, cnt, par)
  if (bv) {
    if (variant == SPH_V3D2) SPH_BIN_COUNT(SPH_V3D2, true);
    else SPH_BIN_COUNT(SPH_V3D4, true);
  } else {
    if (variant == SPH_V2D) SPH_BIN_COUNT(SPH_V2D, false);
    else if (variant == SPH_V3D2) SPH_BIN_COUNT(SPH_V3D2, false);
    else SPH_BIN_COUNT(SPH_V3D4, false);
  }
#undef SPH_BIN_COUNT
}

void launch_bin_table(const BinScratch &bs, uint total_cell, uint *cstart, uint *cend, Counters *cnt,
                      int par, hipStream_t st, bool single, bool keep_err) {
  if (total_cell <= SCAN1_CELLS) {
    k_bin_scan<<<dim3(1), dim3(SCAN1_THREADS), 0, st>>>(bs.ccount, total_cell, cstart, cend, cnt, par,
                                                        single, keep_err);
    return;
  }
  const uint nt = (uint)sph_bin_tiles(total_cell);
  k_bin_tiles<<<dim3(nt), dim3(BLK), 0, st>>>(bs.ccount, total_cell, bs.tmp);
  k_bin_ranges<<<dim3(nt), dim3(BLK), 0, st>>>(bs.ccount, total_cell, bs.tmp, cstart, cend, cnt, par,
                                               single, keep_err);
}

void launch_bin_place(DevState src, const BinScratch &bs, const uint *cstart, const Counters *cnt, uint m,
                      hipStream_t st, uint grid, uint *zero0, uint *zero1, uint per_split, uint zmax) {
  if (m == 0) return;
  k_bin_place<<<bgrid(grid, m), dim3(BLK), 0, st>>>(src.slot, bs.hkey, bs.rank, cstart, cnt, m, bs.bslot,
                                                    zero0, zero1, per_split, zmax);
}

void launch_bin_reorder(DevState src, DevState dst, const BinScratch &bs, const uint *cstart,
                        const uint *cend, uint *skeys, uint *svals, uint *s2p, Counters *cnt, uint m,
                        hipStream_t st, bool all_fields, bool set_m, const BatchView *bv, uint grid,
                        uint *init0, uint *init1, QPosOut qo) {
  if (m == 0) return;
  if (bv)
    k_bin_reorder<true><<<bgrid(grid, m), dim3(BLK), 0, st>>>(
        src, dst, bv->scn, bs.hkey, cstart, cend, bs.bslot, cnt, m, skeys, svals, s2p, all_fields, set_m,
        init0, init1, qo);
  else
    k_bin_reorder<false><<<bgrid(grid, m), dim3(BLK), 0, st>>>(
        src, dst, nullptr, bs.hkey, cstart, cend, bs.bslot, cnt, m, skeys, svals, s2p, all_fields, set_m,
        init0, init1, qo);
}
