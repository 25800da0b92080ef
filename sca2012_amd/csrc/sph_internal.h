// Internal declarations shared by the HIP translation units of libsph_amd.
//
// Device data layout (HBM), per particle, structure-of-arrays and kept in cell order
// (the order of the sorted (hash, slot) list) from the cell-range phase of each step on:
//   pos    float4  x, y, z, w = level (uint bits)        read by every neighbour loop
//   vel    float4  x, y, z, w = 0
//   ev     float4  x, y, z, w = tension (never used by the kernels, kept for AoS I/O)
//   acc    float4  x, y, z, w = surface (|colour-field gradient|)
//   dp     float2  dens, press
//   energy float
//   slot   uint    the particle's index in the reference's Particle array ("slot");
//                  0xffffffff marks a particle removed by merge (dropped at the next sort).
//                  In a batch of scenes the word is scene << 24 | slot within the scene.
// = 80 B per particle; two copies (ping-pong for the reorder).
#ifndef SPH_INTERNAL_H
#define SPH_INTERNAL_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/sph_amd.h"
#include "sph_arith.h"

typedef unsigned int uint;

#define SPH_DEAD 0xffffffffu
#define SPH_EMPTY 0xffffffffu

// Quantised positions (sph_near_q): steps per unit length; per level, minus the squared distance in
// steps below which a pair may interact; the level of the smaller kernel radius, and the mark that
// its particles carry (even; its square is at most the difference of the two squared distances).
struct QParams {
  float scale;
  int neg[2];
  uint mark, mark_level;
};

// Parameters as a by-value kernel argument (no __constant__ global, so contexts are
// independent). Index [0] = large particles (level 1), [1] = small (level 2).
struct DevParams {
  int variant, dim, nsplit;
  float world[3];
  float radius[2], kernel[2], mass[2];
  float cell_size;
  uint ncell[3];
  uint total_cell;
  uint cell_base;  // first global cell of this scene (0 for a single scene)
  float gravity[3];
  float wall_damping, rest_density, gas_constant, time_step, viscosity, surface_tension;
  float co_surface, co_energy, split_criteria, merge_criteria;
  float poly6[2], spiky[2], visco[2], grad[2], lapc[2], k2[2], k6[2], poly6_radius[2];
  float radius2[2];
  float visco_k6[2];  // visco / h^6, the per-level factor of the viscosity kernel
  float sqrt_kernel[2];
  uint nd[3];
  uint tot_dens;
  float den_size;
  float sph_pos[3][3], sph_radius[3], sph_damping[3];
  int push_left, push_right, use_cylinder, mouse;
  float extern_force[2], extern_click[2], extern_len, extern_coe;
  float surf_coef, dens_eps;
  uint cap;
  uint dens_mul;
  // RN(1/x) of the pair terms' constant divisors, for sph_div_mk / sph_div_rn (sph_arith.h)
  float rcp_k6[2], rcp_kernel[2], rcp_sqrt_kernel[2];
  // 1 when the force pair term (spiky*(h-r)^2)/h^6 of both levels meets sph_div_mk's
  // preconditions for every pair (checked on the host from the parameters)
  int k6_fast;
  // 1 when h and sqrt(h) of both levels lie within [2^-20, 2^20] (sph_div_rn's divisors)
  int kernel_div_fast;
  // 1 when every particle's energy kernel length h and sqrt(h) are exactly 1 (3D: the large
  // level's, which both levels use; 2D: both levels'), so x/h and x/sqrt(h) equal x
  int energy_unit;
  QParams q;  // quantised positions (struct Aux: qpos)
};

// Per-step per-particle factors written by the density kernel for the force kernel.
// Per-particle factors of the force pair terms, written by the density kernel, with the
// particle's ev: what the force kernel reads of a neighbour besides its position, as one
// 48-byte record (3 float4) per particle:
//   vpd.x vpd.y ev.x ev.y | gr_0 lc_0 ev.z - | gr_1 lc_1 ev.z -    (2D: vpd.x vpd.y ev.x ev.y)
// with vpd = (m/dens, press/dens^2), gr_L = ((-grad_L) m)/dens and lc_L = (lapc_L m)/dens
// for L = large (0), small (1): a receiver of level L reads the first part and part 1 + L.
// erec, ez: what the energy kernel reads of a neighbour, (pos.x, pos.y, vel.x, vel.y) and pos.z
// after integration, written by the integrate kernel (the velocity's z never reaches the energy).
// nbl (optional): the force kernel's interacting pairs, written by the density kernel,
// which walks the same candidates in the same order: entries packed as
// (offset index << 27) | j in visiting order, four to a 16-byte group, group g of
// particle i at ((uint4 *)nbl)[g * nbl_stride + i] (group-major, so a wave's loads of a
// group are one contiguous run); nbl_cnt[i] entries. A count above SPH_NBL_K means the
// list overflowed (the entries past SPH_NBL_K are not stored) and the force kernel walks
// the cells itself for that particle's wave.
// qpos: the positions in steps of 1/q.scale, modulo 2^16, x | y << 16 and z | mark << 16
// (sph_near_q; the mark of a particle of the smaller kernel, else 0): what the
// one-thread density and energy kernels read of a candidate before its position. Written wherever
// the current positions are: by the reorder, by the integrate kernel and by launch_make_erec.
#define SPH_NBL_K 128u
struct Aux {
  float4 *frec;
  float4 *erec;
  float *ez = nullptr;
  uint2 *qpos = nullptr;
  uint *nbl = nullptr;
  uint *nbl_cnt = nullptr;
  uint nbl_stride = 0;
  // which form of the neighbour kernels runs (choose_forms): several lanes per particle
  // (sph_fine.hip) or one thread (sph_kernels.hip)
  bool fine_density = false, fine_force = false, fine_energy = false;

  // For n live particles of a scene or of a batch's scenes together. Several lanes per
  // particle shorten the chain of dependent loads and cost more instructions, so density and
  // energy are chosen by whether n threads fill the GPU. Measured (one thread -> several
  // lanes, us): density, a falling dam 3D-2 36k 28.9 -> 24.5, 47k 29.2 -> 27.6, 55k 29.2 -> 29.6,
  // 64k 29.2 -> 32.0, an adaptive one 24k 35.0 -> 25.0, 45k 38.3 -> 34.3; a collision 3D-4 43k
  // 49.3 -> 54.5, 53k 66.7 -> 62.5, 64k 61.6 -> 73.7. The two meet near 53k; the line lies at 66k
  // because a rollout chooses by its bound, 65,536 entries for 32^3 particles of which half live
  // at first (36k still: 28.1 -> 24.0). 2D 20k 14 -> 12, 37k
  // 15 -> 15. Energy 3D-2 65k 63 -> 53, 93k 78 -> 69, 128k 101 -> 91, 330k 112 -> 123; 3D-4 76k
  // 108 -> 73, 124k 124 -> 103; 2D 67k 19 -> 16. Force evaluates the same pairs either way, with
  // one pair's registers instead of
  // four: 3D-2 25k 36 -> 15, 498k 107 -> 91; 3D-4 506k 219 -> 134, 1.7M 501 -> 392, 4.2M
  // shrinking to 2M 732 -> 717; 2D 66k 15 -> 13, 264k 24 -> 30; in a batch, whose lanes each
  // load their scene's parameters, 126k 49 -> 39, 400k 41 -> 52. Above the 3D line of a single
  // scene either is the faster: a young dam 6.9M 475 -> 534, falling 8.6M 1118 -> 1039, adaptive
  // 12.0M 1332 -> 1198, a collision 3D-4 6.7M 1509 -> 1419, 9.0M 2212 -> 1798.
  void choose_forms(int variant, bool batch, uint n) {
    const bool d3 = variant != SPH_V2D;
    fine_density = n <= (d3 ? 66000u : 32000u);
    fine_energy = n <= (d3 ? 180000u : 128000u);
    fine_force = n <= (d3 ? (batch ? 150000u : 6000000u) : 100000u);
  }
  // the forms as bits (a captured step depends on them)
  uint forms() const {
    return (fine_density ? 1u : 0u) | (fine_force ? 2u : 0u) | (fine_energy ? 4u : 0u);
  }
};

// where a kernel that writes positions also puts the quantised ones (struct Aux: qpos), if q is
// given; a batch's steps come from its parameter table
struct QPosOut {
  uint2 *q = nullptr;
  QParams Q = {};
  const DevParams *Ptab = nullptr;
};

struct DevState {
  float4 *pos, *vel, *ev, *acc;
  float2 *dp;
  float *energy;
  uint *slot;
};

// Device-resident counters (the step runs without host round trips).
struct Counters {
  uint n;         // live particles
  uint m;         // physical entries (live + removed, until the next sort)
  uint n_pre;     // live count before split (the cell lists cover [0, n_pre))
  uint s_req;     // split parents flagged
  uint s_done;    // split parents split (capacity policy)
  uint groups;    // merge groups
  uint err;       // bit 0: particle outside the grid
  uint ntri;      // triangles emitted by marching cubes
  uint scan_total;  // of launch_pack_live
  uint nmc;  // non-empty marching cubes
  uint m_in;     // entries at the start of the step (m as the step found it)
  uint err2[2];  // domain errors of the step being binned, by step parity (sph_bins.hip)
  uint pad[3];
};

// The counters as a kernel at the end of a step's stream work writes them to pinned host memory,
// with the number of such reports so far: the host polls that number instead of copying the
// counters and synchronising the stream (8 launches and the wait 58 -> 35 us).
struct Report {
  Counters c;
  uint seq;
};
void launch_report(const Counters *cnt, uint *seq, Report *host, hipStream_t st);

// Entries [a, a + na) and [b, b + nb) of the state arrays
struct Span {
  uint a = 0, na = 0, b = 0, nb = 0;
};

// Batches of scenes (one step over many independent scenes): scene s owns the global cells
// [cell_base_s, cell_base_s + total_cell_s) and the dense slot range [first_s, first_s + n_s)
// of the sort input. SceneCnt is its device-resident bookkeeping.
#define SPH_SCENE_SHIFT 24
#define SPH_LOCAL_MASK 0xffffffu
#define SPH_MAX_SCENES 256u  // capacities stay below 0xffffff, so no slot word is SPH_DEAD

struct SceneCnt {
  uint n;          // live particles (updated by split and compaction)
  uint n_pre;      // live particles at the start of the step
  uint first;      // dense start of the scene's slots in the sort input (pre-split)
  uint r0;         // split parents flagged of the scenes before this one
  uint s_req;      // split parents flagged
  uint s_done;     // split parents split (capacity policy)
  uint done_base;  // split parents of the scenes before this one
  uint first2;     // dense start of the scene's slots after split
  uint a0;         // entries removed from the scenes before this one
  uint groups;     // merge groups
  uint err;        // bit 0: particle outside the scene's grid
  uint pad[5];
};

struct BatchView {
  const DevParams *Ptab;  // per-scene parameters (cell_base, cap set)
  SceneCnt *scn;
  uint n_scenes;
  uint total_cell;        // cells of all scenes
};

// ---------------------------------------------------------------------------------------
// XCD-aware block order. The dispatcher hands workgroups to the 8 XCDs round-robin
// (block b to XCD b mod 8), and each XCD has its own L2. Particles are stored in cell
// order, so consecutive blocks are spatial neighbours; this bijection gives XCD x one
// contiguous run of the grid's blocks instead, and the neighbour data a block reads is
// then mostly in its own XCD's L2. A pure permutation of the work: results do not change.
// ---------------------------------------------------------------------------------------
#define SPH_NXCD 8u
__device__ inline uint xcd_block(uint b, uint nb) {
  const uint x = b % SPH_NXCD, k = b / SPH_NXCD;
  const uint q = nb / SPH_NXCD, r = nb % SPH_NXCD;
  return x * q + (x < r ? x : r) + k;
}

// ---------------------------------------------------------------------------------------
// fp32 exp and the reference's wavelet, identical bits on host and device.
// exp: Cody & Waite (1980) argument reduction t = k ln2 + r (ln2 split into a head with
// trailing zero bits and a tail), degree-7 Taylor polynomial of e^r on |r| <= ln2/2 by
// Horner's rule, then scaling by 2^k through the exponent field. Every operation is a
// single IEEE binary32 op in fixed order; the library is compiled without contraction.
// ---------------------------------------------------------------------------------------
__host__ __device__ inline float sph_scale2(float p, int k) {
  if (k > 127) {
    p *= 0x1p127f;
    k -= 127;
  } else if (k < -126) {
    p *= 0x1p-126f;
    k += 126;
    if (k < -126) {
      p *= 0x1p-126f;
      k += 126;
    }
  }
  union { uint u; float f; } s;
  s.u = (uint)(k + 127) << 23;
  return p * s.f;
}

__host__ __device__ inline float sph_expf(float t) {
  if (t != t) return t;
  if (t > 88.75f) return __builtin_huge_valf();
  if (t < -104.0f) return 0.0f;
  const float inv_ln2 = 0x1.715476p+0f;
  const float ln2_hi = 0x1.62e4p-1f;
  const float ln2_lo = 0x1.7f7d1cp-20f;
  float kf = __builtin_rintf(t * inv_ln2);
  float r = (t - kf * ln2_hi) - kf * ln2_lo;
  float p = 0x1.a01a02p-13f;
  p = p * r + 0x1.6c16c2p-10f;
  p = p * r + 0x1.111112p-7f;
  p = p * r + 0x1.555556p-5f;
  p = p * r + 0x1.555556p-3f;
  p = p * r + 0x1p-1f;
  p = p * r + 1.0f;
  p = p * r + 1.0f;
  return sph_scale2(p, (int)kf);
}

// sph_expf for |t| < ln2/2: the reduction above gives k = 0 and r = t exactly and the scale
// is a multiplication by 1, so the polynomial alone returns the same bits.
__host__ __device__ inline float sph_expf_small(float t) {
  float p = 0x1.a01a02p-13f;
  p = p * t + 0x1.6c16c2p-10f;
  p = p * t + 0x1.111112p-7f;
  p = p * t + 0x1.555556p-5f;
  p = p * t + 0x1.555556p-3f;
  p = p * t + 0x1p-1f;
  p = p * t + 1.0f;
  p = p * t + 1.0f;
  return p;
}

// The wavelet for |x| <= 1 (every call site: |x| = |dx|/h with dx a component of a pair
// separation shorter than h), where the exp argument lies in [-0.125, 0].
__host__ __device__ inline float sph_wavelet_unit(float x) {
  const float A = 0x1.3a0156p-1f;
  const float ln_b = 0x1.fffff6p-1f;
  float xx = x * x;
  float b = xx / 4.0f - 1.0f;
  float y = (-xx) / 8.0f;
  return (A * b) * sph_expf_small(y * ln_b);
}

// Entries j .. j+3 of a cell's (or list's) run [.., e), j < e: entries past the end are
// replaced by the run's last entry (in bounds, the same cache line) and the caller skips
// their terms, so a run is walked in groups of four to its end, without a one-by-one tail
// loop.
__device__ inline void sph_group4(const float4 *__restrict__ pos, uint j, uint e, float4 q[4]) {
  const uint l = e - 1;
  q[0] = pos[j];
  q[1] = pos[min(j + 1, l)];
  q[2] = pos[min(j + 2, l)];
  q[3] = pos[min(j + 3, l)];
}

// The same four entries through a buffer resource over the array's first n entries
// (n < 2^28): a load past n returns zeros (the hardware range check) instead of faulting,
// so a run's last group needs no clamping (the caller skips the terms past the run's end,
// and an entry between the run's end and n is a valid particle, merely unused); the four
// loads share one address register with immediate offsets.
__device__ inline __amdgpu_buffer_rsrc_t sph_rsrc(const float4 *a, uint n) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float4 *>(a), (short)0, (int)(n * 16u),
                                           0x00020000);  // gfx9 raw-buffer word 3
}
__device__ inline void sph_group4(__amdgpu_buffer_rsrc_t r, uint j, float4 q[4]) {
  const uint off = j * 16u;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, off + 16u * k, 0, 0);
    q[k] = make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]),
                       __uint_as_float(v[3]));
  }
}

__device__ inline __amdgpu_buffer_rsrc_t sph_rsrc8(const uint2 *a, uint n) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint2 *>(a), (short)0, (int)(n * 8u), 0x00020000);
}

// Quantised positions. A candidate's squared distance is first formed in whole steps of 1/q.scale
// (a power of two; the larger kernel radius is 2048 to 4096 steps): two packed 16-bit subtractions
// and two dot products instead of eight fp32 operations, from 8 bytes instead of 16. A rounded
// coordinate is within half a step, so a difference is within one, and a pair whose fp32 distance
// is below h has a squared step distance below (h q.scale (1 + 1e-5) + 2)^2 = -q.neg (sqrt(3) < 2;
// 1e-5 covers the rounding of the fp32 distance). Coordinates are kept modulo 2^16 and sums modulo
// 2^32, so a candidate far away may pass as well: every one that passes is tested in fp32, and none
// that interacts is lost. Coordinates beyond 2^31 steps saturate.
// The fourth 16-bit place makes the distance of a pair of the smaller kernel's level count for
// more, where the pair's reach is the larger of the two radii: with a particle of that level at 0
// there, a candidate of the same level (at the mark) gains mark^2, the difference of the two
// thresholds; a particle at mark / 2 sees candidates of both levels alike.
typedef short sph_short2 __attribute__((ext_vector_type(2)));
__host__ __device__ inline uint sph_qcoord(float x, float scale) {
  // NaN and everything below -2^31 become -2^31, what is above the last float below 2^31 that float
  const float s = __builtin_fminf(__builtin_fmaxf(__builtin_rintf(x * scale), -0x1p31f), 0x1.fffffep30f);
  return (uint)(int)s & 0xffffu;
}
// of a position with its level in w
__host__ __device__ inline uint2 sph_qpos(float x, float y, float z, uint level, const QParams &Q) {
  uint2 q;
  q.x = sph_qcoord(x, Q.scale) | sph_qcoord(y, Q.scale) << 16;
  q.y = sph_qcoord(z, Q.scale) | ((level == 1u ? 0u : 1u) == Q.mark_level ? Q.mark << 16 : 0u);
  return q;
}
// what a particle of level index L compares its candidates with: reach of a pair max(h_i, h_j)
// (either) or h of level index L alone
struct QSelf {
  uint2 q;
  int neg;
};
__host__ __device__ inline QSelf sph_qself(uint2 q, int L, bool either, const QParams &Q) {
  const bool marked = either && (uint)L == Q.mark_level;
  const uint half = marked ? 0u : Q.mark / 2u;
  QSelf r;
  r.q = q;
  r.q.y = (q.y & 0xffffu) | half << 16;
  const int far = Q.neg[0] < Q.neg[1] ? Q.neg[0] : Q.neg[1];
  // half^2 less, which every candidate gains
  r.neg = (either ? far : Q.neg[L]) + (int)(half * half) * -1;
  return r;
}
// negative when the pair may interact
__device__ inline int sph_near_q(const QSelf &a, uint bx, uint by) {
  const sph_short2 d = __builtin_bit_cast(sph_short2, a.q.x) - __builtin_bit_cast(sph_short2, bx);
  const sph_short2 e = __builtin_bit_cast(sph_short2, a.q.y) - __builtin_bit_cast(sph_short2, by);
  return __builtin_amdgcn_sdot2(d, d, __builtin_amdgcn_sdot2(e, e, a.neg, false), false);
}

// Correctly rounded sqrtf for finite x >= 2^-96: the hardware estimate, then whichever
// neighbour one ulp away the two fma residuals select (the correction the compiler's IEEE
// sqrtf applies; its extra input scaling and zero/infinity fix-ups concern only x below
// 2^-96 and non-finite x).
__device__ inline float sph_sqrt_normal(float x) {
  float s = __builtin_amdgcn_sqrtf(x);
  const float sm = __uint_as_float(__float_as_uint(s) - 1u);
  const float sp = __uint_as_float(__float_as_uint(s) + 1u);
  const float rm = __builtin_fmaf(-sm, s, x);
  const float rp = __builtin_fmaf(-sp, s, x);
  if (rm <= 0.0f) s = sm;
  if (rp > 0.0f) s = sp;
  return s;
}

// SPH-3D-2/sph_system.cu:11-16: 2/(PI^.25 (3 sigma)^.5) (x^2/sigma^2 - 1) EXP^(-x^2/(2 sigma^2)),
// sigma = 2, PI = 3.141592f, EXP = 2.718281f; EXP^y = exp(y ln EXP).
__host__ __device__ inline float sph_wavelet(float x) {
  const float A = 0x1.3a0156p-1f;    // 2 / (float(PI^0.25) * sqrtf(6))
  const float ln_b = 0x1.fffff6p-1f; // float(ln 2.718281f)
  float xx = x * x;
  float b = xx / 4.0f - 1.0f;
  float y = (-xx) / 8.0f;
  return (A * b) * sph_expf(y * ln_b);
}

// ---------------------------------------------------------------------------------------
// Launch wrappers (sph_kernels.hip / sph_prims.hip)
// ---------------------------------------------------------------------------------------
struct SortScratch {
  uint *keys_alt, *vals_alt;  // ping-pong partners
  uint *tile_hist;            // sph_sort_hist_elems(n)
};

size_t sph_scan_tmp_elems(size_t n);
size_t sph_sort_hist_elems(size_t n);  // histogram entries for a sort of n keys

// Exclusive scan of in[0..*n_dev) (host upper bound n_max) into out; total -> *total_dev.
void sph_exclusive_scan(const uint *in, uint *out, const uint *n_dev, uint n_max, uint *total_dev,
                        uint *tmp, hipStream_t st);
// Stable LSD radix sort of keys[0..n) (values = slot index 0..n-1, generated) by the low
// `bits` bits. Result (keys, vals) ends in (*keys_out, *vals_out), which point into
// {keys, vals} or {sc.keys_alt, sc.vals_alt}. n_dev (optional): the key
// count in device memory, n bounding it; grid (optional): persistent histogram and scatter
// launches of that many workgroups.
void sph_radix_sort(uint *keys, uint *vals, uint n, int bits, SortScratch &sc, uint **keys_out,
                    uint **vals_out, hipStream_t st, const uint *n_dev = nullptr, uint grid = 0);
// Cell order by counting (sph_bins.hip), for grids that a scan over all cells suits.
struct BinScratch {
  uint *ccount;  // entries per cell, all zero between steps
  uint *hkey;    // cell of each entry
  uint *rank;    // arrival rank of each entry in its cell
  uint *bslot;   // slots by cell, in arrival order
  uint *tmp;     // tile sums, sph_bin_tiles(total_cell)
};
// Bits by slot (a batch: by dense slot) and by entry, for split and merge; sph_bit_words words each
struct SlotBits {
  uint *split;     // slot -> split decided
  uint *dead;      // slot -> removed by a merge
  uint *qual;      // entry in cell order -> qualifies for merging
  uint *toff;      // sph_bit_tiles: scan of the tiles' counts (sph_slots.hip)
  uint *scan_tmp;  // for that scan
};
size_t sph_bit_words(size_t n);
size_t sph_bit_tiles(size_t n);
// Counting or radix sort for n particles on total_cell cells. The scan reads and writes 20
// bytes per cell (4M cells: 18 us, about what the sort's extra launches take). Hash, sort, table
// and reorder against counting: 14k particles on 13,824 cells 33 -> 19 us, 498k on 262,144 cells
// 88 -> 76 us.
bool sph_use_bins(size_t total_cell, size_t n);
size_t sph_bin_tiles(size_t total_cell);
// m bounds the entries (the device's cnt->m counts them). Single scenes: the kernels also start
// the step's counters and collect domain errors under the step's parity `par`, which alternates
// from step to step.
void launch_bin_count(int variant, const DevParams &P, DevState src, const BinScratch &bs,
                      Counters *cnt, uint m, int par, hipStream_t st, const BatchView *bv = nullptr,
                      uint grid = 0);
void launch_bin_table(const BinScratch &bs, uint total_cell, uint *cstart, uint *cend, Counters *cnt,
                      int par, hipStream_t st, bool single = true, bool keep_err = false);
// zero0, zero1 (optional): bit arrays to clear, for the m entries and for (1 + per_split) m, at most
// zmax words
void launch_bin_place(DevState src, const BinScratch &bs, const uint *cstart, const Counters *cnt, uint m,
                      hipStream_t st, uint grid = 0, uint *zero0 = nullptr, uint *zero1 = nullptr,
                      uint per_split = 0, uint zmax = 0);
// skeys, svals: the sorted keys and slots; s2p: slot -> place; set_m: also cnt->m = cnt->n;
// init0, init1 (optional): SPH_DEAD for every particle
void launch_bin_reorder(DevState src, DevState dst, const BinScratch &bs, const uint *cstart,
                        const uint *cend, uint *skeys, uint *svals, uint *s2p, Counters *cnt, uint m,
                        hipStream_t st, bool all_fields, bool set_m = true,
                        const BatchView *bv = nullptr, uint grid = 0, uint *init0 = nullptr,
                        uint *init1 = nullptr, QPosOut qo = {});
void sph_fill_u32(uint *p, uint value, size_t n, hipStream_t st);
// cstart[0..n) = SPH_EMPTY and cend[0..n) = 0 in one launch
void sph_fill_cells(uint *cstart, uint *cend, size_t n, hipStream_t st);
// the cells that launch_cell_bounds(skeys, n, ncell, ...) wrote, back to the fill values
void sph_reset_cells(const uint *skeys, uint n, uint ncell, uint *cstart, uint *cend,
                     hipStream_t st);

// `bv` (batches only) selects the kernels that read the scene of each particle from its
// slot word and its parameters from bv->Ptab.
// Launch shapes of the per-item kernels: `n_dev` (optional) is a device word holding the
// item count, and `n` then only bounds it (the buffers' size); `grid` (optional) is a
// persistent grid of that many workgroups, each looping over blocks of 256 items, else the
// grid has one workgroup per block of n. A launch with both is independent of the host's
// view of the counts, as a captured graph needs.
void launch_hash(int variant, const DevParams &P, DevState s, const uint *cnt_m, uint m_max,
                 uint *keys, uint *slot2phys, Counters *cnt, hipStream_t st,
                 const BatchView *bv = nullptr, uint grid = 0);
void launch_cell_bounds(const uint *skeys, uint n, uint ncell, uint *cstart, uint *cend,
                        hipStream_t st, const uint *n_dev = nullptr, uint grid = 0);
// set_m: also cnt->m = cnt->n (removed entries are gone once reordered)
// all_fields == false: acc, dp and energy are not carried (a step recomputes them)
void launch_reorder(DevState src, DevState dst, const uint *svals, const uint *slot2phys, uint n,
                    uint *slot2phys_new, hipStream_t st, Counters *set_m = nullptr,
                    bool all_fields = true, const uint *n_dev = nullptr, uint grid = 0,
                    QPosOut qo = {});
// The neighbour kernels (density, force, energy) and merge run one thread per particle (or
// cell, or sorted key) on a grid sized by n, which bounds the device count n_dev if given.
// density with a.nbl: also the force kernel's pair lists; force with use_nbl: reads them
// (they must come from a density pass over the same state, cell lists and parameters).
void launch_density(int variant, const DevParams &P, DevState s, Aux a, const uint *cstart,
                    const uint *cend, uint n, hipStream_t st, const BatchView *bv = nullptr,
                    const uint *n_dev = nullptr);
// Pair-list lengths that a program can set; `cfg` indexes the force kernel's. The energy kernel
// keeps cells, not pairs, in its lanes' rings and is the same for every energy length.
constexpr int kForceLists[3] = {24, 32, 48};
constexpr int kEnergyLists[3] = {16, 24, 32};
constexpr int kForceListDefault = 1, kEnergyListDefault = 0;
// A new context or batch runs a round of 6 tuning steps after its first 8 steps and then
// one every 128 steps (a scene's neighbour counts, and with them the best length, drift).
constexpr uint kTuneRounds = 0xffffffffu, kTuneAfter = 8, kTuneEvery = 128;
constexpr float kTuneMargin = 0.05f;  // a length replaces the one in use when 5% faster
// ... and, in a list-tuning round after the first, when 10% faster: those rounds compare a
// length chosen for the scene against alternatives that are rarely better by more than a
// few percent, so their measurement noise must not move the choice
constexpr float kTuneMarginLater = 0.10f;
void launch_force(int variant, const DevParams &P, DevState s, Aux a, const uint *cstart,
                  const uint *cend, uint n, hipStream_t st, const BatchView *bv = nullptr,
                  int cfg = kForceListDefault, const uint *n_dev = nullptr,
                  bool use_nbl = false);
// and each particle's energy record and quantised position (a.erec, a.ez, a.qpos)
void launch_integrate(int variant, const DevParams &P, DevState s, uint n, hipStream_t st,
                      const BatchView *bv, Aux a, const uint *n_dev = nullptr, uint grid = 0);
// split_bits (optional): also the split decision of each particle (as launch_decide), as bits
// that were clear before; qbits (optional, not with `fine`): also the merge qualification of the
// entries as it stands before the split; a.erec, a.qpos: the energy records and quantised
// positions of the current positions and velocities (written by the integrate kernel, or by
// launch_make_erec)
void launch_energy(int variant, const DevParams &P, DevState s, Aux a, const uint *cstart,
                   const uint *cend, uint n, hipStream_t st, const BatchView *bv,
                   uint *split_bits, uint *qbits, const uint *n_dev = nullptr);
// the same phases in several lanes per particle (launch_density, launch_force and launch_energy
// call these as Aux::choose_forms says)
void launch_density_fine(int variant, const DevParams &P, DevState s, Aux a, const uint *cstart,
                         const uint *cend, uint n, hipStream_t st, const BatchView *bv,
                         const uint *n_dev);
void launch_force_fine(int variant, const DevParams &P, DevState s, Aux a, const uint *cstart,
                       const uint *cend, uint n, hipStream_t st, const BatchView *bv,
                       const uint *n_dev, bool use_nbl);
void launch_energy_fine(int variant, const DevParams &P, DevState s, const uint *cstart,
                        const uint *cend, uint n, hipStream_t st, const BatchView *bv,
                        uint *split_bits, const float4 *erec, const uint *n_dev);
void launch_make_erec(const DevParams &P, DevState s, uint n, Aux a, hipStream_t st,
                      const uint *n_dev = nullptr);
void launch_decide(int variant, const DevParams &P, DevState s, uint n, uint *split_bits, hipStream_t st);
// Split of the flagged ones of the cnt->n_pre (at most n) particles (sph_slots.hip). s2p: slot ->
// entry. A single scene's split also applies the capacity policy to the counters (n, m, s_req,
// s_done); a batch's counters come from launch_batch_split_plan. with_qual: the entries'
// qualification bits are completed; child (optional): entry of a parent -> its first child.
void launch_split(int variant, const DevParams &P, DevState s, uint n, const SlotBits &sb, const uint *s2p,
                  Counters *cnt, hipStream_t st, bool with_qual, const BatchView *bv = nullptr,
                  uint *child = nullptr);
// 2D merge qualification word per cell (bit 0; the entry + 1 of the cell id's particle in
// bits 1..31 when it is listed in that cell)
void launch_merge_q2d(const DevParams &P, DevState s, const uint *slot2phys, const Counters *cnt,
                      const uint *cstart, const uint *cend, uint *q2d, hipStream_t st);
// skeys/nkeys (optional): the step's sorted cell keys; on a grid with more cells than keys
// the merge then runs one thread per key instead of one per cell (same result).
// dead: bits by slot (clear before) that receive the removed entries. qbits (optional): the
// entries' qualification bits, ready (from the energy kernel and the split) or evaluated first,
// one thread per entry, instead of inside each cell's walk (same result)
void launch_merge(int variant, const DevParams &P, DevState s, const uint *cstart,
                  const uint *cend, const uint *q2d, uint *dead, Counters *cnt, hipStream_t st,
                  const BatchView *bv = nullptr, const uint *skeys = nullptr, uint nkeys = 0,
                  const uint *nkeys_dev = nullptr, uint *group_out = nullptr,
                  uint *qbits = nullptr, bool qbits_ready = false);
// Slots of the survivors among the cnt->m (at most m) entries; removed entries become SPH_DEAD.
// A single scene's renumbering also sets the live count. all_slots: s2p maps every slot, else
// those of the n_pre particles before the split.
void launch_renumber(int variant, DevState s, uint m, const SlotBits &sb, const uint *s2p, bool all_slots,
                     Counters *cnt, hipStream_t st, const BatchView *bv = nullptr);
void launch_begin_step(Counters *cnt, hipStream_t st);
// batch bookkeeping (one block each): dense slot starts, split plan, survivor counts
void launch_batch_begin(const BatchView &bv, Counters *cnt, hipStream_t st);
void launch_batch_split_plan(int variant, const BatchView &bv, Counters *cnt, hipStream_t st);
void launch_batch_compact_plan(int variant, const BatchView &bv, Counters *cnt, hipStream_t st);
// move the live entries of [0, m) to the front of dst, in order; *cnt_live = their number
void launch_pack_live(DevState src, DevState dst, uint m, uint *flags, uint *pos, uint *tmp,
                      uint *total_dev, hipStream_t st);
// occ: 2 * sph_occ_words(total_cell) words of scratch for the cell-occupancy bitmap of the
// general (per-voxel) kernel and its 27-cell dilation; unused by the cell-block kernel
inline size_t sph_occ_words(size_t ncell) { return (ncell + 63) / 64 * 2; }
void launch_density_grid(const DevParams &P, DevState s, const uint *cstart, const uint *cend,
                         float *dgrid, bool cell_blocks, hipStream_t st, uint *occ);
void launch_normals(const DevParams &P, const float *dgrid, float *normal3, hipStream_t st);
size_t mc_segments(const DevParams &P);  // z-segments of marching cubes (count/offset entries)
void launch_mc_count(const DevParams &P, const float *dgrid, uint *seg_tri, uint *seg_cube,
                     hipStream_t st);
void launch_mc_list(const DevParams &P, const float *dgrid, const uint *seg_cube,
                    const uint *seg_toff, const uint *seg_coff, uint cap, uint2 *clist,
                    hipStream_t st);
void launch_mc_emit(const DevParams &P, const float *dgrid, const float *normal3, const uint2 *clist,
                    const Counters *cnt, uint max_tri, float *tris, hipStream_t st);
// AoS records -> entries [base, base + n) of s (entry base + i gets slot word slot_or | i). cnt
// (optional): the counters become those of `live` particles in `entries` entries. bv: the scene's
// entries in `old` are removed and the scenes' counters start over
void launch_upload(int variant, const void *aos_dev, uint n, DevState s, uint base, hipStream_t st,
                   Counters *cnt, uint live, uint entries, uint slot_or = 0u, Span old = {},
                   const BatchView *bv = nullptr);
// the first n records (by slot) of the scene with the scene bits `scene` among the entries `at`
void launch_download(int variant, DevState s, Span at, uint n, void *aos_dev, hipStream_t st,
                     uint scene = 0u);
void launch_slot2phys(DevState s, uint m, uint *slot2phys, hipStream_t st);

// Online autotuner of the force kernel's pair-list length, shared by the single-scene context
// and the batch. The length never changes the order in which a particle's terms are summed, so
// the results do not depend on tuning. Tuning starts after `after` steps (a scene's first steps
// are not representative: cold caches, and an adaptive scene grows over its first few steps). A
// round is 12 tuning steps (the first round of a tuning run 6); each runs the force and energy
// kernels once, the force kernel with one candidate length, bracketed by events; the candidates
// take turns in the order 0 1 2 2 1 0 0 1 2 2 1 0, so a cost that drifts linearly from step to
// step (a scene's neighbour counts keep changing) weighs on every candidate alike. The first
// round decides between lengths that differ by 20% or more at a scene's start; the later ones
// compare lengths within a few percent, so each candidate's mean is over four launches (with
// two, launch-to-launch noise made a later round pick a length 9% slower than the one in use).
// After a round the force kernel switches to the candidate with the lowest mean time if it beats
// the length in use by more than kTuneMargin. Rounds repeat every `every` steps, as the best
// length drifts with the neighbour counts (shorter lists win while a scene is sparse).
// What has one form has nothing to choose: the energy kernel at every length, and the force
// kernel while it runs in several lanes per particle (force_counts is false), which keeps no such
// list. Their time stands for every length, and a round without a choice is one timed step if
// no times are there yet, else none, so that steps stay captured.
struct ListTuner {
  static constexpr int kRound = 12;
  static constexpr int kOrder[kRound] = {0, 1, 2, 2, 1, 0, 0, 1, 2, 2, 1, 0};
  int force = kForceListDefault, energy = kEnergyListDefault;
  bool force_counts = true;     // the next step's force kernel has lists (set before each step)
  uint rounds_left = 0, skip = 0, every = 0;
  int steps_left = 0, pos = 0, round_len = 0;
  bool pending = false;         // a tuning step's events are not read yet
  float sum[2][3];              // [force, energy][candidate] total ms over the tuning steps
  int cnt[2][3];
  float best[2][3];             // mean ms per candidate (-1: not measured)
  hipEvent_t ev[2][2] = {};     // [kernel][begin, end]

  bool create() {
    for (auto &k : ev)
      for (auto &e : k)
        if (hipEventCreate(&e) != hipSuccess) return false;
    return true;
  }
  void destroy() {
    for (auto &k : ev)
      for (auto &e : k)
        if (e) (void)hipEventDestroy(e);
  }
  void start(uint rounds, uint after, uint every_steps) {
    rounds_left = rounds;
    round_len = kRound / 2;
    steps_left = rounds ? round_len : 0;
    skip = rounds ? after : 0;
    every = every_steps > (uint)kRound ? every_steps : (uint)kRound;
    pos = 0;
    pending = false;
    clear_sums();
    for (auto &k : best)
      for (float &b : k) b = -1.0f;
  }
  void clear_sums() {
    for (int k = 0; k < 2; k++)
      for (int c = 0; c < 3; c++) {
        sum[k][c] = 0.0f;
        cnt[k][c] = 0;
      }
  }
  // the next step is a tuning step
  bool tuning() const { return steps_left > 0 && skip == 0 && (force_counts || best[0][0] < 0.0f); }
  bool active() const { return steps_left > 0; }
  // pin the lengths (stops tuning); false if a length is not a candidate
  bool set(uint force_len, uint energy_len) {
    int f = -1, e = -1;
    for (int c = 0; c < 3; c++) {
      if ((uint)kForceLists[c] == force_len) f = c;
      if ((uint)kEnergyLists[c] == energy_len) e = c;
    }
    if (f < 0 || e < 0) return false;
    force = f;
    energy = e;
    rounds_left = 0;
    steps_left = 0;
    skip = 0;
    pending = false;
    return true;
  }
  // kernel 0 = force, 1 = energy; launch(cfg) enqueues one run (of the force kernel with that candidate)
  template <class F> void run(int kernel, hipStream_t st, F launch) {
    if (!tuning()) {
      launch(kernel == 0 ? force : energy);
      return;
    }
    (void)hipEventRecord(ev[kernel][0], st);
    launch(kOrder[pos % kRound]);
    (void)hipEventRecord(ev[kernel][1], st);
    pending = true;
  }
  // after the step's synchronisation
  void end_step() {
    if (steps_left == 0) return;
    if (skip > 0) {
      skip--;
      return;
    }
    if (!pending && force_counts) return;
    const int c = kOrder[pos % kRound];
    if (pending)
      for (int k = 0; k < 2; k++) {
        float ms = 0.0f;
        if (hipEventElapsedTime(&ms, ev[k][0], ev[k][1]) != hipSuccess) continue;
        for (int j = 0; j < 3; j++)
          if (j == c || k == 1 || !force_counts) {
            sum[k][j] += ms;
            cnt[k][j] += 1;
          }
      }
    pending = false;
    pos++;
    steps_left = force_counts ? steps_left - 1 : 0;
    if (steps_left > 0) return;
    for (int k = 0; k < 2; k++)
      for (int j = 0; j < 3; j++)
        if (cnt[k][j]) best[k][j] = sum[k][j] / (float)cnt[k][j];
    if (force_counts) {
      const float margin = round_len < kRound ? kTuneMargin : kTuneMarginLater;
      int pick = force;
      for (int j = 0; j < 3; j++)
        if (best[0][j] >= 0.0f && best[0][force] >= 0.0f && best[0][j] < best[0][force] * (1.0f - margin) &&
            best[0][j] < best[0][pick])
          pick = j;
      force = pick;
    }
    rounds_left--;
    if (rounds_left > 0) {  // the next round, `every` steps after this one started
      skip = every - (uint)pos;
      round_len = kRound;
      steps_left = kRound;
      pos = 0;
      clear_sums();
    }
  }
};

// Host-side parameter handling shared by the single-scene context and the batch.
namespace sphhost {
bool valid_variant(int v);
DevParams make_dev_params(int variant, const void *raw, uint cap);
int key_bits(uint total_cell);
size_t sysparam_size(int variant);
size_t particle_size(int variant);
}  // namespace sphhost

#endif
