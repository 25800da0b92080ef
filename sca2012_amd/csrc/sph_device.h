// Device helpers shared by the step's kernel files (sph_kernels.hip, sph_fine.hip, sph_bins.hip,
// sph_prims.hip): work-item mapping, the variants' compile-time properties, cell arithmetic, the
// neighbour order and block scans.
#ifndef SPH_DEVICE_H
#define SPH_DEVICE_H

#include "sph_internal.h"

namespace {


constexpr int BLK = 256;

// Work-item count: the device count when given (clamped to the host bound, which sizes the
// buffers), else the host count.
__device__ inline uint dev_count(const uint *n_dev, uint n_host) {
  return n_dev ? min(*n_dev, n_host) : n_host;
}

// Items [0, n) in blocks of BLK: block vb of nvb = ceil(n / BLK) is handled by workgroup
// vb mod gridDim.x. A plain launch has one workgroup per block and runs one iteration; a
// persistent launch (a fixed grid sized for the GPU, a multiple of the 8 XCDs) loops over
// the blocks. With XCD the blocks map XCD-contiguously (xcd_block): workgroup w runs on XCD
// w mod 8, and so does every block w + k * gridDim.x it takes.
template <bool XCD, class F> __device__ inline void for_each_item(uint n, F &&item) {
  const uint nvb = (n + BLK - 1) / BLK;
  for (uint vb = blockIdx.x; vb < nvb; vb += gridDim.x) {
    const uint i = (XCD ? xcd_block(vb, nvb) : vb) * BLK + threadIdx.x;
    if (i < n) item(i);
  }
}

// One thread per item for the kernels whose blocks cost unevenly (the neighbour loops):
// the launch has one workgroup per block of a bound of n (the host's count, or in a graph
// the buffer's size while n is read on the device), the blocks past n exit at once and the
// hardware dispatcher balances the rest; block vb runs on XCD vb mod 8 and takes block
// xcd_block(vb, nvb). False for a thread with no item.
__device__ inline bool one_item(uint n, uint &i) {
  const uint nvb = (n + BLK - 1) / BLK;
  if (blockIdx.x >= nvb) return false;
  i = xcd_block(blockIdx.x, nvb) * BLK + threadIdx.x;
  return i < n;
}

template <int V> struct VT {
  static constexpr int dim = V == SPH_V2D ? 2 : 3;
  static constexpr int nsplit = V == SPH_V3D4 ? 4 : 2;
  static constexpr int nnb = dim == 2 ? 9 : 27;
};

// Neighbour offsets in the reference's order (SPH-3D-2/sph_system.cu:456-562; 2D :383-408):
// within each z layer (z, z-1, z+1) the in-plane order is
// (0,0) (-1,-1) (-1,0) (0,-1) (1,1) (1,0) (0,1) (1,-1) (-1,1).
__device__ constexpr int kDX[9] = {0, -1, -1, 0, 1, 1, 0, 1, -1};
__device__ constexpr int kDY[9] = {0, -1, 0, -1, 1, 0, 1, -1, 1};
__device__ constexpr int kDZ[3] = {0, -1, 1};

__device__ inline int lvl_index(float w) { return __float_as_uint(w) == 1u ? 0 : 1; }

// Parameters of a particle's scene: the by-value block of a single scene, or the batch
// table entry named by the scene bits of its slot word.
template <bool B>
__device__ inline const DevParams &scene_params(const DevParams &P0,
                                                const DevParams *__restrict__ Ptab, uint w) {
  if constexpr (B) return Ptab[w >> SPH_SCENE_SHIFT];
  else return P0;
}

// entry q of the quantised positions (w: its slot word)
template <bool B> __device__ inline void put_qpos(const QPosOut &qo, uint q, uint w, const float4 &p) {
  if (!qo.q) return;
  qo.q[q] = sph_qpos(p.x, p.y, p.z, __float_as_uint(p.w), B ? qo.Ptab[w >> SPH_SCENE_SHIFT].q : qo.Q);
}

// calc_grid_pos (SPH-3D-2/sph_system.cu:18-27): (uint)floor(p / cell_size); false when the
// coordinate is outside [0, ncell) or NaN.
template <int V>
__device__ inline bool cell_of(const DevParams &P, float x, float y, float z, uint c[3]) {
  float q0 = floorf(x / P.cell_size);
  float q1 = floorf(y / P.cell_size);
  bool ok = (q0 >= 0.0f) && (q0 < (float)P.ncell[0]) && (q1 >= 0.0f) && (q1 < (float)P.ncell[1]);
  c[0] = ok ? (uint)q0 : 0u;
  c[1] = ok ? (uint)q1 : 0u;
  c[2] = 0u;
  if (VT<V>::dim == 3) {
    float q2 = floorf(z / P.cell_size);
    bool ok2 = (q2 >= 0.0f) && (q2 < (float)P.ncell[2]);
    c[2] = ok2 ? (uint)q2 : 0u;
    ok = ok && ok2;
  }
  return ok;
}

// neighbor_status (SPH-3D-2/sph_system.cu:564-652) and calc_grid_hash (:29-32)
template <int V>
__device__ inline bool neighbor_cell(const DevParams &P, int o, const uint c[3], uint &h) {
  const int g = o % 9, dx = kDX[g], dy = kDY[g], dz = kDZ[o / 9];
  if (dx == -1 && c[0] == 0) return false;
  if (dx == 1 && c[0] == P.ncell[0] - 1) return false;
  if (dy == -1 && c[1] == 0) return false;
  if (dy == 1 && c[1] == P.ncell[1] - 1) return false;
  if (VT<V>::dim == 3) {
    if (dz == -1 && c[2] == 0) return false;
    if (dz == 1 && c[2] == P.ncell[2] - 1) return false;
  }
  h = P.cell_base + (c[2] + (uint)dz) * P.ncell[0] * P.ncell[1] + (c[1] + (uint)dy) * P.ncell[0] +
      (c[0] + (uint)dx);
  return true;
}

// (dx+1) | (dy+1) << 2 of the nine in-plane offsets, 4 bits each, in offset order,
// derived at compile time from the same in-plane order as kDX/kDY.
constexpr unsigned long long make_off_xy() {
  constexpr int dx[9] = {0, -1, -1, 0, 1, 1, 0, 1, -1};
  constexpr int dy[9] = {0, -1, 0, -1, 1, 0, 1, -1, 1};
  unsigned long long v = 0;
  for (int g = 0; g < 9; g++)
    v |= (unsigned long long)((dx[g] + 1) | ((dy[g] + 1) << 2)) << (4 * g);
  return v;
}
constexpr unsigned long long kOffXY = make_off_xy();
static_assert(kOffXY == 0x8296a1405ull, "in-plane offset table");

// Particle range [s, e) of neighbour cell o (o wave-uniform, loop not unrolled); empty
// when the reference's neighbor_status disables the cell or it holds no particle.
template <int V>
__device__ inline void nb_range(const DevParams &P, int o, const uint c[3],
                                const uint *__restrict__ cstart, const uint *__restrict__ cend,
                                uint &s, uint &e) {
  const int g = o % 9, zl = o / 9;
  const int code = (int)((kOffXY >> (4 * g)) & 0xfull);
  const int dx = (code & 3) - 1, dy = (code >> 2) - 1;
  const int dz = zl == 0 ? 0 : (zl == 1 ? -1 : 1);
  s = e = 0;
  if (dx == -1 && c[0] == 0) return;
  if (dx == 1 && c[0] == P.ncell[0] - 1) return;
  if (dy == -1 && c[1] == 0) return;
  if (dy == 1 && c[1] == P.ncell[1] - 1) return;
  if (VT<V>::dim == 3) {
    if (dz == -1 && c[2] == 0) return;
    if (dz == 1 && c[2] == P.ncell[2] - 1) return;
  }
  const uint h = P.cell_base + (c[2] + (uint)dz) * P.ncell[0] * P.ncell[1] +
                 (c[1] + (uint)dy) * P.ncell[0] + (c[0] + (uint)dx);
  const uint st = cstart[h];
  const uint en = cend[h];  // issued with the start load; 0 for an empty cell
  if (st == SPH_EMPTY) return;
  s = st;
  e = en;
}

// Interacting-pair lists: entry = (offset index << 27) | particle index, kept in LDS
// column-major ([k][thread]) so a wave's accesses hit distinct banks.
// The list length only moves the drain points, never the order in which a particle's
// pairs are summed, so every length gives the same bits (sph_internal.h: kForceLists).
__device__ inline uint pack_entry(int o, uint j) { return ((uint)o << 27) | j; }

// Split decision of the particle with slot word w: its bit by slot (a batch: by dense slot, and
// the scene's count of flagged parents, one atomic per wave where the wave's are of one scene).
template <bool B>
__device__ inline void flag_split(bool split, uint w, uint *__restrict__ split_bits, SceneCnt *scn) {
  if (!split) return;
  uint d = w;
  if constexpr (B) {
    const uint sc = w >> SPH_SCENE_SHIFT;
    d = scn[sc].first + (w & SPH_LOCAL_MASK);
    const uint sc0 = (uint)__builtin_amdgcn_readfirstlane((int)sc);
    const unsigned long long here = __ballot(true), same = __ballot(sc == sc0);
    if (here != same) atomicAdd(&scn[sc].s_req, 1u);
    else if ((threadIdx.x & 63u) == (uint)__builtin_ctzll(here))
      atomicAdd(&scn[sc].s_req, (uint)__popcll(here));
  }
  atomicOr(&split_bits[d >> 5], 1u << (d & 31u));
}

__device__ inline uint wave_incl_scan(uint x, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  return x;
}

// Exclusive scan of one value per thread across the block; returns the block total.
__device__ inline uint block_excl_scan(uint x, uint *lds_waves, uint &total) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  uint inc = wave_incl_scan(x, lane);
  if (lane == 63) lds_waves[w] = inc;
  __syncthreads();
  uint before = 0, tot = 0;
  for (int k = 0; k < (int)(blockDim.x >> 6); k++) {
    uint v = lds_waves[k];
    if (k < w) before += v;
    tot += v;
  }
  __syncthreads();
  total = tot;
  return before + inc - x;
}

}  // namespace

#endif
