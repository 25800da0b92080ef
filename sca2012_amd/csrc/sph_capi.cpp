// C ABI of libsph_amd (declared in include/sph_amd.h): parameter derivation, the context
// that owns every device buffer, the phase entry points and the whole step.
//
// Per-step device work (one HIP stream, no host round trip until the end of the step):
//   particles counted into cells -> cell table -> place -> reorder into cell order
//   (sph_bins.hip; a sparse grid, and the phase calls: hash -> radix sort -> cell ranges +
//   reorder) -> density -> force -> integrate -> [density grid -> normals -> marching cubes] ->
//   energy -> [split] -> [merge -> renumber survivors]
// Counts that change inside the step (after split and merge) stay on the device; kernels
// read them and are launched over host-side upper bounds. A step that repeats is launched as one
// captured graph, and a kernel at its end reports the counters into pinned memory that the host
// polls (graph_step, sync).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdio>
#include <cstring>
#include <new>
#include <vector>

#include "sph_internal.h"

static_assert(sizeof(SphSysParam3D) == 296, "SysParam 3D layout (SPH-3D-2/sph_param.h)");
static_assert(sizeof(SphParticle3D) == 72, "Particle 3D layout (SPH-3D-2/sph_system.h)");
static_assert(sizeof(SphSysParam2D) == 200, "SysParam 2D layout (SPH-2D/sph_param.h)");
static_assert(sizeof(SphParticle2D) == 56, "Particle 2D layout (SPH-2D/sph_system.h)");
static_assert(offsetof(SphSysParam3D, sphere1) == 204, "SysParam 3D sphere offset");
static_assert(offsetof(SphSysParam3D, flag0) == 292, "SysParam 3D flag offset");
static_assert(offsetof(SphSysParam2D, extern_force) == 168, "SysParam 2D extern_force offset");

#define SPH_VERSION "sph_amd 0.1 gfx950"

namespace {

const float kPI = 3.141592f;  // SPH-3D-2/sph_header.h:22

bool valid_variant(int v) { return v == SPH_V2D || v == SPH_V3D2 || v == SPH_V3D4; }

// Kernel constants of the reference constructor (SPH-3D-2/sph_system.cpp:63-84;
// SPH-2D/sph_system.cpp:19-41). pow(float, int) is evaluated in double, as C++11 does.
void derive_kernel_constants(float h, float &poly6, float &spiky, float &visco, float &grad,
                             float &lapc, float &k2, float &k6) {
  poly6 = (float)(315.0f / (64.0f * kPI * std::pow((double)h, 9)));
  spiky = (float)(-45.0f / (kPI * std::pow((double)h, 6)));
  visco = (float)(45.0f / (kPI * std::pow((double)h, 6)));
  grad = (float)(-945.0f / (32.0f * kPI * std::pow((double)h, 9)));
  lapc = (float)(-945.0f / (8.0f * kPI * std::pow((double)h, 9)));
  k2 = h * h;
  k6 = (float)std::pow((double)h, 6);
}

void derive3(SphSysParam3D &s) {
  s.cell_size = s.large_kernel;
  s.row_cell = (uint)std::ceil(s.world_width / s.cell_size);
  s.col_cell = (uint)std::ceil(s.world_height / s.cell_size);
  s.len_cell = (uint)std::ceil(s.world_length / s.cell_size);
  s.total_cell = s.row_cell * s.col_cell * s.len_cell;
  s.world_width = s.row_cell * s.cell_size;
  s.world_height = s.col_cell * s.cell_size;
  s.world_length = s.len_cell * s.cell_size;
  derive_kernel_constants(s.large_kernel, s.large_poly6, s.large_spiky, s.large_visco,
                          s.large_grad_poly6, s.large_lapc_poly6, s.large_kernel_2, s.large_kernel_6);
  derive_kernel_constants(s.small_kernel, s.small_poly6, s.small_spiky, s.small_visco,
                          s.small_grad_poly6, s.small_lapc_poly6, s.small_kernel_2, s.small_kernel_6);
  s.large_poly6_radius = (float)(315.0f / (64.0f * kPI * std::pow((double)s.large_radius, 9)));
  s.small_poly6_radius = (float)(315.0f / (64.0f * kPI * std::pow((double)s.small_radius, 9)));
  if (s.dens_mul == 0) s.dens_mul = 4;
  s.den_size = s.cell_size / s.dens_mul;
  s.row_dens = s.row_cell * s.dens_mul + 1;
  s.col_dens = s.col_cell * s.dens_mul + 1;
  s.len_dens = s.len_cell * s.dens_mul + 1;
  s.tot_dens = s.row_dens * s.col_dens * s.len_dens;
}

void derive2(SphSysParam2D &s) {
  derive_kernel_constants(s.large_kernel, s.large_poly6, s.large_spiky, s.large_visco,
                          s.large_grad_poly6, s.large_lapc_poly6, s.large_kernel2, s.large_kernel6);
  derive_kernel_constants(s.small_kernel, s.small_poly6, s.small_spiky, s.small_visco,
                          s.small_grad_poly6, s.small_lapc_poly6, s.small_kernel2, s.small_kernel6);
  s.cell_size = s.large_kernel;
  s.row_cell = (uint)std::ceil(s.world_width / s.cell_size);
  s.col_cell = (uint)std::ceil(s.world_depth / s.cell_size);
  s.total_cell = s.row_cell * s.col_cell;
  s.world_width = s.row_cell * s.cell_size;
  s.world_depth = s.col_cell * s.cell_size;
}

// SPH-3D-2/sph_system.cpp:6-229 and SPH-3D-4/sph_system.cpp:6-230
void defaults3(int variant, SphSysParam3D &s) {
  std::memset(&s, 0, sizeof(s));
  const bool v4 = variant == SPH_V3D4;
  s.max_particle = 1000000;
  s.world_width = v4 ? 48.0f : 32.0f;
  s.world_height = v4 ? 24.0f : 16.0f;
  s.world_length = v4 ? 24.0f : 16.0f;
  s.large_radius = v4 ? 1.2f : 1.0f;
  s.small_radius = 0.8f;
  s.large_kernel = v4 ? 1.2f : 1.0f;
  s.large_mass = 1.0f;
  s.small_kernel = v4 ? 1.0f : 0.9f;
  s.small_mass = v4 ? 0.25f : 0.5f;
  s.gravity = {0.0f, v4 ? -4.0f : -5.0f, 0.0f};
  s.wall_damping = -0.6f;
  s.rest_density = v4 ? 0.5f : 1.0f;
  s.gas_constant = 1.0f;
  s.time_step = 0.1f;
  s.viscosity = v4 ? 1.0f : 3.0f;
  s.surface_tension = 0.8f;
  s.co_surface = v4 ? 1.5f : 1.0f;
  s.co_energy = 1.0f;
  s.split_criteria = v4 ? 1.0f : 1.2f;
  s.merge_criteria = v4 ? 0.6f : 0.4f;
  s.dens_mul = 4;
  s.sphere1 = {{11.0f, 3.0f, 4.0f}, 2.0f, 1.0f};
  s.sphere2 = {{11.0f, 3.0f, 12.0f}, 2.0f, 1.0f};
  s.sphere3 = {{18.0f, 3.0f, 8.0f}, 2.0f, 1.0f};
  s.split_energy = 0.8f;
  s.merge_energy = 0.02f;
  derive3(s);
}

// SPH-2D/sph_system.cpp:5-146
void defaults2(SphSysParam2D &s) {
  std::memset(&s, 0, sizeof(s));
  s.max_particle = 100000;
  s.world_width = 32.0f;
  s.world_depth = 32.0f;
  s.large_mass = 1.0f;
  s.small_mass = 0.5f;
  s.large_kernel = 1.0f;
  s.small_kernel = 0.9f;
  s.large_radius = 1.0f;
  s.small_radius = 0.8f;
  s.gravity = {0.0f, -4.5f};
  s.wall_damping = -0.6f;
  s.rest_density = 2.0f;
  s.gas_constant = 1.0f;
  s.viscosity = 2.0f;
  s.time_step = 0.1f;
  s.surface_normal = 0.5f;
  s.co_surface = 0.8f;
  s.co_energy = 1.0f;
  s.thresh_split = 0.7f;
  s.thresh_merge = 0.04f;
  s.extern_len = 2.0f;
  s.extern_coe = 1.0f;
  derive2(s);
}

DevParams make_dev_params(int variant, const void *raw, uint cap) {
  DevParams P;
  std::memset(&P, 0, sizeof(P));
  P.variant = variant;
  P.cap = cap;
  if (variant == SPH_V2D) {
    const SphSysParam2D &s = *(const SphSysParam2D *)raw;
    P.dim = 2;
    P.nsplit = 2;
    P.world[0] = s.world_width; P.world[1] = s.world_depth; P.world[2] = 0.0f;
    P.radius[0] = s.large_radius; P.radius[1] = s.small_radius;
    P.kernel[0] = s.large_kernel; P.kernel[1] = s.small_kernel;
    P.mass[0] = s.large_mass; P.mass[1] = s.small_mass;
    P.cell_size = s.cell_size;
    P.ncell[0] = s.row_cell; P.ncell[1] = s.col_cell; P.ncell[2] = 1;
    P.total_cell = s.total_cell;
    P.gravity[0] = s.gravity.x; P.gravity[1] = s.gravity.y; P.gravity[2] = 0.0f;
    P.wall_damping = s.wall_damping; P.rest_density = s.rest_density;
    P.gas_constant = s.gas_constant; P.time_step = s.time_step; P.viscosity = s.viscosity;
    P.surface_tension = s.surface_normal;
    P.co_surface = s.co_surface; P.co_energy = s.co_energy;
    P.split_criteria = s.thresh_split; P.merge_criteria = s.thresh_merge;
    P.poly6[0] = s.large_poly6; P.poly6[1] = s.small_poly6;
    P.spiky[0] = s.large_spiky; P.spiky[1] = s.small_spiky;
    P.visco[0] = s.large_visco; P.visco[1] = s.small_visco;
    P.grad[0] = s.large_grad_poly6; P.grad[1] = s.small_grad_poly6;
    P.lapc[0] = s.large_lapc_poly6; P.lapc[1] = s.small_lapc_poly6;
    P.k2[0] = s.large_kernel2; P.k2[1] = s.small_kernel2;
    P.k6[0] = s.large_kernel6; P.k6[1] = s.small_kernel6;
    P.mouse = s.force_waiting ? 1 : 0;
    P.extern_force[0] = s.extern_force.x; P.extern_force[1] = s.extern_force.y;
    P.extern_click[0] = s.extern_click.x; P.extern_click[1] = s.extern_click.y;
    P.extern_len = s.extern_len; P.extern_coe = s.extern_coe;
    P.surf_coef = 0.04f;  // SPH-2D/sph_system.cu:770
    P.dens_eps = 1e-12f;  // EXT2, SPH-2D/sph_system.cu:8, :320
  } else {
    const SphSysParam3D &s = *(const SphSysParam3D *)raw;
    P.dim = 3;
    P.nsplit = variant == SPH_V3D4 ? 4 : 2;
    P.world[0] = s.world_width; P.world[1] = s.world_height; P.world[2] = s.world_length;
    P.radius[0] = s.large_radius; P.radius[1] = s.small_radius;
    P.kernel[0] = s.large_kernel; P.kernel[1] = s.small_kernel;
    P.mass[0] = s.large_mass; P.mass[1] = s.small_mass;
    P.cell_size = s.cell_size;
    P.ncell[0] = s.row_cell; P.ncell[1] = s.col_cell; P.ncell[2] = s.len_cell;
    P.total_cell = s.total_cell;
    P.gravity[0] = s.gravity.x; P.gravity[1] = s.gravity.y; P.gravity[2] = s.gravity.z;
    P.wall_damping = s.wall_damping; P.rest_density = s.rest_density;
    P.gas_constant = s.gas_constant; P.time_step = s.time_step; P.viscosity = s.viscosity;
    P.surface_tension = s.surface_tension;
    P.co_surface = s.co_surface; P.co_energy = s.co_energy;
    P.split_criteria = s.split_criteria; P.merge_criteria = s.merge_criteria;
    P.poly6[0] = s.large_poly6; P.poly6[1] = s.small_poly6;
    P.spiky[0] = s.large_spiky; P.spiky[1] = s.small_spiky;
    P.visco[0] = s.large_visco; P.visco[1] = s.small_visco;
    P.grad[0] = s.large_grad_poly6; P.grad[1] = s.small_grad_poly6;
    P.lapc[0] = s.large_lapc_poly6; P.lapc[1] = s.small_lapc_poly6;
    P.k2[0] = s.large_kernel_2; P.k2[1] = s.small_kernel_2;
    P.k6[0] = s.large_kernel_6; P.k6[1] = s.small_kernel_6;
    P.poly6_radius[0] = s.large_poly6_radius; P.poly6_radius[1] = s.small_poly6_radius;
    P.nd[0] = s.row_dens; P.nd[1] = s.col_dens; P.nd[2] = s.len_dens;
    P.tot_dens = s.tot_dens;
    P.den_size = s.den_size;
    P.dens_mul = s.dens_mul;
    const SphSphere *sp[3] = {&s.sphere1, &s.sphere2, &s.sphere3};
    for (int k = 0; k < 3; k++) {
      P.sph_pos[k][0] = sp[k]->pos.x; P.sph_pos[k][1] = sp[k]->pos.y; P.sph_pos[k][2] = sp[k]->pos.z;
      P.sph_radius[k] = sp[k]->radius; P.sph_damping[k] = sp[k]->damping;
    }
    if (variant == SPH_V3D4) {
      P.push_left = s.flag0; P.push_right = s.flag1; P.use_cylinder = s.flag2;
    } else {
      P.push_left = s.flag0; P.push_right = 0; P.use_cylinder = s.flag1;
    }
    P.surf_coef = variant == SPH_V3D4 ? 0.02f : 0.1f;  // 3D-4 :1136, 3D-2 :1129
    P.dens_eps = 0.0001f;
  }
  P.radius2[0] = P.radius[0] * P.radius[0];
  P.radius2[1] = P.radius[1] * P.radius[1];
  P.visco_k6[0] = P.visco[0] / P.k6[0];
  P.visco_k6[1] = P.visco[1] / P.k6[1];
  P.sqrt_kernel[0] = std::sqrt(P.kernel[0]);  // pow(kernel, 0.5f)
  P.sqrt_kernel[1] = std::sqrt(P.kernel[1]);
  P.k6_fast = 1;
  P.kernel_div_fast = 1;
  for (int l = 0; l < 2; l++) {  // after sqrt_kernel
    P.rcp_k6[l] = sph_rcp_rn(P.k6[l]);
    P.rcp_kernel[l] = sph_rcp_rn(P.kernel[l]);
    P.rcp_sqrt_kernel[l] = sph_rcp_rn(P.sqrt_kernel[l]);
    if (!sph_k6_div_fast(P.spiky[l], P.kernel[l], P.k6[l])) P.k6_fast = 0;
    for (float d : {P.kernel[l], P.sqrt_kernel[l]})
      if (!(d >= 0x1p-20f && d <= 0x1p20f)) P.kernel_div_fast = 0;
  }
  // steps for the quantised distance test (sph_near_q), from the longer kernel
  const double hq = std::sqrt((double)std::max(P.k2[0], P.k2[1]));
  P.q = QParams{0.0f, {-1, -1}, 0u, 0u};  // every position the same: no pair is ruled out
  if (hq > 1e-30 && hq < 1e30 && P.k2[0] >= 0.0f && P.k2[1] >= 0.0f) {
    P.q.scale = (float)std::exp2(std::floor(std::log2(4096.0 / hq)));
    for (int l = 0; l < 2; l++) {
      const double r = std::sqrt((double)P.k2[l]) * P.q.scale * (1.0 + 1e-5) + 2.0;
      P.q.neg[l] = -(int)std::ceil(r * r);
    }
    P.q.mark_level = P.k2[1] <= P.k2[0] ? 1u : 0u;
    P.q.mark = (uint)std::sqrt((double)std::abs(P.q.neg[0] - P.q.neg[1])) & ~1u;
  }
  P.energy_unit = 1;
  for (int l = 0; l < (P.dim == 3 ? 1 : 2); l++)
    if (!(P.kernel[l] == 1.0f && P.sqrt_kernel[l] == 1.0f)) P.energy_unit = 0;
  return P;
}

// The cell-block density-grid kernel assumes that the voxels dens_mul*c + 1 ... dens_mul*c +
// dens_mul along each axis are exactly those the reference maps to cell c,
// floor((float)v / (float)n_dens * (float)n_cell) (SPH-3D-2/sph_system.cu:1946-1948). This
// checks it for every voxel index, in the same fp32 arithmetic.
bool dgrid_cell_blocks_exact(const DevParams &P) {
  if (P.dim != 3 || P.dens_mul != 4) return false;
  for (int a = 0; a < 3; a++) {
    if (P.nd[a] != P.ncell[a] * P.dens_mul + 1) return false;
    for (uint v = 1; v < P.nd[a]; v++) {
      const uint c = (uint)std::floor((float)v / (float)P.nd[a] * (float)P.ncell[a]);
      if (c != (v - 1) / P.dens_mul) return false;
    }
  }
  return true;
}

int key_bits(uint total_cell) {
  int b = 1;
  while (b < 32 && ((uint64_t)1 << b) < (uint64_t)total_cell) b++;
  return b;
}

}  // namespace

namespace {
// Polls of a report before the host waits for the stream instead (about 0.3 ms)
constexpr uint kReportPolls = 10000;
// Steps with the same launches before they are captured, and captured steps that are kept
constexpr uint kGraphAfter = 3;
constexpr size_t kGraphsMax = 16;
}  // namespace

namespace sphhost {
bool valid_variant(int v) { return ::valid_variant(v); }
DevParams make_dev_params(int variant, const void *raw, uint cap) {
  return ::make_dev_params(variant, raw, cap);
}
int key_bits(uint total_cell) { return ::key_bits(total_cell); }
size_t sysparam_size(int variant) {
  return variant == SPH_V2D ? sizeof(SphSysParam2D) : sizeof(SphSysParam3D);
}
size_t particle_size(int variant) {
  return variant == SPH_V2D ? sizeof(SphParticle2D) : sizeof(SphParticle3D);
}
}  // namespace sphhost

struct SphCtx {
  int variant = 0;
  unsigned char raw[296];
  size_t raw_size = 0;
  DevParams P;
  uint cap = 0, max_tri = 0;
  hipStream_t st = nullptr;
  DevState cur{}, alt{};
  Aux aux{};
  std::vector<void *> allocs;
  uint *keys = nullptr, *vals = nullptr;
  SortScratch sc{};
  BinScratch bins{};
  int par = 0;  // parity of the step (counting path)
  uint *s2p_hash = nullptr, *s2p_cell = nullptr;
  uint *cstart = nullptr, *cend = nullptr;
  SlotBits sb{};
  uint *newslot = nullptr, *q2d = nullptr;
  uint *scan_tmp = nullptr;
  Counters *cnt = nullptr;
  uint *rep_seq = nullptr;       // reports made, on the device
  Report *rep = nullptr;         // the last report (pinned host memory) and its device address
  Report *rep_dev = nullptr;
  uint rep_want = 0;             // reports that were launched
  float *dgrid = nullptr, *normal3 = nullptr, *tris = nullptr;
  uint *cube_count = nullptr, *cube_off = nullptr;  // per z-segment: triangles, their offsets
  uint *seg_cube = nullptr, *seg_coff = nullptr;    // per z-segment: non-empty cubes, offsets
  uint2 *clist = nullptr;                           // non-empty cubes (id, first triangle)
  bool dgrid_cells = false;                         // cell-block density-grid kernel applies
  uint *occ = nullptr;                              // cell occupancy bits and their dilation
  size_t ncube = 0;
  unsigned char *aos_dev = nullptr;
  uint *skeys = nullptr, *svals = nullptr;
  uint n = 0, m = 0, n_pre = 0;
  uint n_sorted = 0, n_flagged = 0, n_status = 0;
  bool hashed = false, sorted = false, lists_valid = false, merged = false, compacted = false;
  bool qual_ready = false;  // the step's energy kernel wrote sb.qual
  // aux.erec, ez and qpos hold the current positions and velocities, in the current parameters' steps
  bool erec_ok = false;
  // aux.nbl holds the force pairs of the current state, cell lists and parameters (the
  // density kernel writes them; anything else that runs invalidates them)
  bool nbl_ok = false;
  // Cell tables: cells_keys/cells_nkeys are the sorted keys they were built from (valid
  // until the next hash or sort overwrites them); cells_clean = every entry holds its fill
  // value. On a sparse grid the next build resets only the cells those keys wrote.
  const uint *cells_keys = nullptr;
  uint cells_nkeys = 0;
  bool cells_clean = false;
  int kbits = 1;
  hipError_t last_err = hipSuccess;
  // profiling
  uint32_t prof_mask = 0;  // phases timed with events (bit k = phase k)
  std::vector<hipEvent_t> ev_pool;
  struct Pending { int phase; hipEvent_t a, b; };
  std::vector<Pending> pending;
  double prof_ms[SPH_P_COUNT] = {0};
  uint64_t prof_n[SPH_P_COUNT] = {0};
  int open_phase = -1;
  hipEvent_t open_ev = nullptr;

  ListTuner tune;  // pair-list length of the force kernel

  // Captured steps (graph_step): everything a step's launches depend on but the device's state
  struct StepKey {
    uint bound, flags, forms, list, buffers;
    bool operator==(const StepKey &o) const {
      return bound == o.bound && flags == o.flags && forms == o.forms && list == o.list &&
             buffers == o.buffers;
    }
  };
  struct StepGraph {
    StepKey key;
    uint uses;
    uint64_t last;
    hipGraphExec_t exec;  // null until the step has run kGraphAfter times
  };
  StepGraph graphs[kGraphsMax];  // the first n_graphs
  size_t n_graphs = 0;
  uint64_t graph_clock = 0;
  bool graphs_work = true;    // false once a capture has failed
  bool flipped = false;       // cur is the second state buffer
  const uint *nd = nullptr;   // during a capture: the live count on the device, n and m bound it

  ~SphCtx() {
    if (st) (void)hipStreamSynchronize(st);
    tune.destroy();
    for (auto &p : pending) {
      (void)hipEventDestroy(p.a);
      (void)hipEventDestroy(p.b);
    }
    for (auto e : ev_pool) (void)hipEventDestroy(e);
    for (void *p : allocs) (void)hipFree(p);
    for (size_t k = 0; k < n_graphs; k++)
      if (graphs[k].exec) (void)hipGraphExecDestroy(graphs[k].exec);
    if (rep) (void)hipHostFree(rep);
    if (st) (void)hipStreamDestroy(st);
  }

  template <class T> bool alloc(T *&p, size_t count) {
    void *q = nullptr;
    if (count == 0) count = 1;
    if (hipMalloc(&q, count * sizeof(T)) != hipSuccess) return false;
    allocs.push_back(q);
    p = (T *)q;
    return true;
  }

  bool alloc_state(DevState &s) {
    return alloc(s.pos, cap) && alloc(s.vel, cap) && alloc(s.ev, cap) && alloc(s.acc, cap) &&
           alloc(s.dp, cap) && alloc(s.energy, cap) && alloc(s.slot, cap);
  }

  hipEvent_t take_event() {
    if (!ev_pool.empty()) {
      hipEvent_t e = ev_pool.back();
      ev_pool.pop_back();
      return e;
    }
    hipEvent_t e = nullptr;
    (void)hipEventCreate(&e);
    return e;
  }
  void pbegin(int phase) {
    if (!((prof_mask >> phase) & 1u)) return;
    open_phase = phase;
    open_ev = take_event();
    (void)hipEventRecord(open_ev, st);
  }
  void pend() {
    if (open_phase < 0) return;
    hipEvent_t b = take_event();
    (void)hipEventRecord(b, st);
    pending.push_back({open_phase, open_ev, b});
    open_phase = -1;
  }
  void collect() {
    for (auto &p : pending) {
      float ms = 0.0f;
      if (hipEventElapsedTime(&ms, p.a, p.b) == hipSuccess) {
        prof_ms[p.phase] += ms;
        prof_n[p.phase] += 1;
      }
      ev_pool.push_back(p.a);
      ev_pool.push_back(p.b);
    }
    pending.clear();
  }

  int fail(hipError_t e) {
    last_err = e;
    return SPH_EHIP;
  }
  // Wait for the stream's work; the counters stay as the host knows them. An error that was there
  // before (of a launch, or left in this thread by other code) is returned, but not before the
  // work is done: copies to or from the caller's memory may be among it.
  int drain() {
    hipError_t err = hipGetLastError();
    const hipError_t e = hipStreamSynchronize(st);
    if (err == hipSuccess) err = e;
    if (err != hipSuccess) return fail(err);
    collect();
    return SPH_OK;
  }
  // Read the counters once the stream's work is done, collect timings. Returns an SPH status.
  // reported: the work ended with a report kernel, counted in rep_want where it was launched. The
  // host polls the report's number for a while, about what a small scene's step takes, and then
  // waits for the stream; a stream that fails, or ends without the report, ends the wait there.
  // An error that was there before is returned after the counters are read, so that they and the
  // number of reports stay those of the device.
  int sync(bool reported = false) {
    hipError_t err = hipGetLastError();
    if (!reported) {
      launch_report(cnt, rep_seq, rep_dev, st);
      const hipError_t e = hipGetLastError();
      if (e == hipSuccess) rep_want++;
      else if (err == hipSuccess) err = e;
    }
    const bool events = !pending.empty() || tune.pending;  // read below or by the caller
    auto there = [&] { return __atomic_load_n(&rep->seq, __ATOMIC_ACQUIRE) == rep_want; };
    bool done = false;
    for (uint k = 0; !events && err == hipSuccess && !done && k < kReportPolls; k++) {
      done = there();
      __builtin_ia32_pause();
    }
    if (!done) {
      const hipError_t e = hipStreamSynchronize(st);
      if (e != hipSuccess || !there()) {  // the work failed
        rep_want = rep->seq;
        return fail(err != hipSuccess ? err : e != hipSuccess ? e : hipErrorUnknown);
      }
    }
    collect();
    n = rep->c.n;
    m = rep->c.m;
    return err == hipSuccess ? SPH_OK : fail(err);
  }

  // ---- enqueue-only phase bodies ----
  // before the sorted keys behind the cell tables are overwritten
  void retire_cells() {
    if (!cells_keys) return;
    if ((size_t)cells_nkeys * 16 < P.total_cell) {  // sparse: undo the written cells only
      sph_reset_cells(cells_keys, cells_nkeys, P.total_cell, cstart, cend, st);
      cells_clean = true;
    }
    cells_keys = nullptr;
  }
  void q_hash() {
    nbl_ok = false;
    retire_cells();
    launch_begin_step(cnt, st);
    pbegin(SPH_P_HASH);
    launch_hash(variant, P, cur, cnt ? &cnt->m : nullptr, m, keys, s2p_hash, cnt, st);
    pend();
  }
  void q_sort() {
    nbl_ok = false;
    retire_cells();
    pbegin(SPH_P_SORT);
    sph_radix_sort(keys, vals, n, kbits, sc, &skeys, &svals, st);
    n_sorted = n;
    pend();
  }
  // in_step: the step's density, force and energy kernels follow, so the reorder leaves out
  // the fields they overwrite
  QPosOut qout() const { return QPosOut{aux.qpos, P.q, nullptr}; }
  void q_cells(bool in_step = false) {
    nbl_ok = false;
    pbegin(SPH_P_CELLS);
    if (!cells_clean) sph_fill_cells(cstart, cend, P.total_cell, st);
    launch_cell_bounds(skeys, n, P.total_cell, cstart, cend, st);
    cells_keys = skeys;
    cells_nkeys = n;
    cells_clean = false;
    pend();
    pbegin(SPH_P_REORDER);
    launch_reorder(cur, alt, svals, s2p_hash, n, s2p_cell, st, cnt, !in_step, nullptr, 0,
                   qout());  // and m = n
    pend();
    erec_ok = false;
    std::swap(cur, alt);
    flipped = !flipped;
  }
  // hash, sort, cell ranges and reorder of a step: by counting where the grid suits it. The bits
  // that the step's split and merge set start clear.
  // After a step that found particles outside the grid the sort takes over: those particles go to
  // cell 0, and an entry's place in its cell costs a pass over the cell (sph_bins.hip).
  bool by_counting() const { return bins.ccount && !rep->c.err && sph_use_bins(P.total_cell, n); }
  void q_bin_step(bool do_split, bool do_merge) {
    if (!nd && !by_counting()) {
      q_hash();
      q_sort();
      q_cells(true);
      if (do_split) sph_fill_u32(sb.split, 0u, sph_bit_words(n), st);
      if (do_merge) sph_fill_u32(sb.dead, 0u, sph_bit_words(grown(n)), st);
      return;
    }
    nbl_ok = false;
    erec_ok = false;
    cells_keys = nullptr;  // every table entry is written again
    cells_clean = false;
    par ^= 1;
    skeys = sc.keys_alt;
    svals = sc.vals_alt;
    n_sorted = n;
    pbegin(SPH_P_HASH);
    launch_bin_count(variant, P, cur, bins, cnt, m, par, st);
    pend();
    pbegin(SPH_P_CELLS);
    launch_bin_table(bins, P.total_cell, cstart, cend, cnt, par, st);
    pend();
    pbegin(SPH_P_SORT);
    launch_bin_place(cur, bins, cstart, cnt, m, st, 0, do_split ? sb.split : nullptr,
                     do_merge ? sb.dead : nullptr, variant == SPH_V3D4 ? 3u : 1u,
                     (uint)sph_bit_words(cap));
    pend();
    pbegin(SPH_P_REORDER);
    launch_bin_reorder(cur, alt, bins, cstart, cend, skeys, svals, s2p_cell, cnt, m, st, false, true, nullptr,
                       0, nullptr, nullptr, qout());
    pend();
    std::swap(cur, alt);
    flipped = !flipped;
  }
  // entries that a split of k particles can leave
  uint grown(uint k) const {
    const uint64_t most = (uint64_t)k * (variant == SPH_V3D4 ? 4u : 2u);
    return most < cap ? (uint)most : std::max(cap, k);
  }
  void q_density(bool in_step = false) {
    pbegin(SPH_P_DENSITY);
    if (!nd) aux.choose_forms(variant, false, n);
    if (!in_step && !aux.fine_density) launch_make_erec(P, cur, n, aux, st);  // for qpos
    launch_density(variant, P, cur, aux, cstart, cend, n, st, nullptr, nd);
    pend();
    nbl_ok = true;
  }
  // tuned: a step may run the autotuner's candidates (the phase calls use its choice)
  void q_force(bool tuned = false) {
    pbegin(SPH_P_FORCE);
    const bool use = nbl_ok;
    if (!nd) aux.choose_forms(variant, false, n);
    auto go = [&](int c) {
      launch_force(variant, P, cur, aux, cstart, cend, n, st, nullptr, c, nd, use);
    };
    if (tuned) tune.run(0, st, go);
    else go(tune.force);
    pend();
  }
  void q_integrate() {
    nbl_ok = false;
    pbegin(SPH_P_INTEGRATE);
    launch_integrate(variant, P, cur, n, st, nullptr, aux, nd);
    pend();
    erec_ok = true;
  }
  // do_split, do_merge (a step): the energy kernel also makes the split decisions (q_split(true)
  // follows), and its one-thread form the merge qualification
  void q_energy(bool tuned = false, bool do_split = false, bool do_merge = false) {
    pbegin(SPH_P_ENERGY);
    if (!erec_ok) {  // not straight after integrate: records from the current state
      launch_make_erec(P, cur, n, aux, st);
      erec_ok = true;
    }
    if (!nd) aux.choose_forms(variant, false, n);
    qual_ready = do_merge && !aux.fine_energy;
    auto go = [&](int) {
      launch_energy(variant, P, cur, aux, cstart, cend, n, st, nullptr, do_split ? sb.split : nullptr,
                    qual_ready ? sb.qual : nullptr, nd);
    };
    if (tuned) tune.run(1, st, go);
    else go(tune.energy);
    pend();
  }
  // in_step: the decisions and the slot map are there
  void q_split(bool in_step = false) {
    nbl_ok = false;
    erec_ok = false;
    pbegin(SPH_P_SPLIT);
    const uint *s2p = s2p_cell;
    if (!in_step) {
      sph_fill_u32(sb.split, 0u, sph_bit_words(n), st);
      launch_decide(variant, P, cur, n, sb.split, st);
      launch_slot2phys(cur, m, newslot, st);
      s2p = newslot;
    }
    launch_split(variant, P, cur, n, sb, s2p, cnt, st, in_step && qual_ready);
    n_flagged = n;
    pend();
  }
  void q_merge(bool in_step = false) {
    nbl_ok = false;
    erec_ok = false;
    pbegin(SPH_P_MERGE);
    if (variant == SPH_V2D) launch_merge_q2d(P, cur, s2p_cell, cnt, cstart, cend, q2d, st);
    // all of them: a split may still come before compact, and its children's slots follow
    if (!in_step) sph_fill_u32(sb.dead, 0u, sph_bit_words(cap), st);
    // a step in several lanes per particle leaves the qualification to each cell's walk
    launch_merge(variant, P, cur, cstart, cend, q2d, sb.dead, cnt, st, nullptr, skeys, n_sorted,
                 nd, nullptr, in_step && !qual_ready ? nullptr : sb.qual, in_step);
    pend();
  }
  void q_compact(bool in_step = false) {
    nbl_ok = false;
    pbegin(SPH_P_COMPACT);
    if (!in_step) launch_slot2phys(cur, m, newslot, st);
    launch_renumber(variant, cur, in_step ? grown(n) : m, sb, in_step ? s2p_cell : newslot, !in_step, cnt,
                    st);  // and n = survivors
    pend();
  }
  void q_dgrid() {
    pbegin(SPH_P_DGRID);
    launch_density_grid(P, cur, cstart, cend, dgrid, dgrid_cells, st, occ);
    pend();
  }
  void q_normals() {
    pbegin(SPH_P_NORMALS);
    launch_normals(P, dgrid, normal3, st);
    pend();
  }
  void q_mc() {
    pbegin(SPH_P_MC);
    launch_mc_count(P, dgrid, cube_count, seg_cube, st);
    sph_exclusive_scan(cube_count, cube_off, nullptr, (uint)ncube, &cnt->ntri, scan_tmp, st);
    sph_exclusive_scan(seg_cube, seg_coff, nullptr, (uint)ncube, &cnt->nmc, scan_tmp, st);
    launch_mc_list(P, dgrid, seg_cube, cube_off, seg_coff, max_tri, clist, st);
    launch_mc_emit(P, dgrid, normal3, clist, cnt, max_tri, tris, st);
    pend();
  }

  void q_step(uint flags) {
    const bool do_split = (flags & SPH_STEP_SPLIT) != 0, do_merge = (flags & SPH_STEP_MERGE) != 0;
    q_bin_step(do_split, do_merge);
    q_density(true);
    q_force(true);
    q_integrate();
    if ((flags & SPH_STEP_MC) && P.dim == 3 && dgrid) {
      q_dgrid();
      q_normals();
      q_mc();
    }
    q_energy(true, do_split, do_merge);
    if (do_split) q_split(true);
    if (do_merge) {
      q_merge(true);
      q_compact(true);
    }
  }

  void drop_graphs() {
    if (n_graphs == 0) return;
    (void)hipStreamSynchronize(st);
    for (size_t k = 0; k < n_graphs; k++)
      if (graphs[k].exec) (void)hipGraphExecDestroy(graphs[k].exec);
    n_graphs = 0;
  }
  // The step as one captured graph, its report included, when it has run kGraphAfter times with
  // the same launches (a capture takes longer than a step; a scene that is stepped a few times
  // never pays for one). The launches are sized by a power of two above the particle and entry
  // counts and read the counts on the device. Steps of sparse grids (whose host state decides how
  // the cell tables are cleared), timed steps and steps with one-step forces are launched one by
  // one. Returns false if the step is still to be launched.
  bool graph_step(uint flags) {
    if (!graphs_work || prof_mask || tune.tuning() || !by_counting() || P.push_left || P.push_right || P.mouse)
      return false;
    uint bound = 1024;
    while (bound < std::max(n, m) && bound < cap) bound *= 2;
    bound = std::min(bound, cap);
    const StepKey key{bound, flags & 7u, aux.forms(), tune.force_counts ? (uint)tune.force : 0u,
                      (flipped ? 1u : 0u) | (par ? 2u : 0u)};
    StepGraph *const all = graphs, *end = all + n_graphs;
    StepGraph *g = std::find_if(all, end, [&](const StepGraph &x) { return x.key == key; });
    if (g == end) {
      if (n_graphs < kGraphsMax) {
        n_graphs++;
      } else {  // the one unused for longest goes
        g = std::min_element(all, end, [](const StepGraph &a, const StepGraph &b) { return a.last < b.last; });
        if (g->exec) {
          (void)hipStreamSynchronize(st);
          (void)hipGraphExecDestroy(g->exec);
        }
      }
      *g = StepGraph{key, 0u, 0u, nullptr};
    }
    g->last = ++graph_clock;
    if (!g->exec) {
      if (++g->uses <= kGraphAfter) return false;
      // the capture records the step without running it: what it leaves in the host's state is undone
      struct Host {
        DevState cur, alt;
        bool flipped, nbl_ok, erec_ok, qual_ready, cells_clean;
        int par;
        uint n, m, n_sorted, n_flagged, cells_nkeys;
        uint *skeys, *svals;
        const uint *cells_keys;
      } h{cur, alt, flipped, nbl_ok, erec_ok, qual_ready, cells_clean, par, n, m, n_sorted, n_flagged,
          cells_nkeys, skeys, svals, cells_keys};
      hipGraph_t rec = nullptr;
      hipError_t e = hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal);
      if (e == hipSuccess) {
        n = m = bound;
        nd = &cnt->n_pre;
        q_step(flags);
        launch_report(cnt, rep_seq, rep_dev, st);
        nd = nullptr;
        e = hipStreamEndCapture(st, &rec);
      }
      cur = h.cur, alt = h.alt, flipped = h.flipped, nbl_ok = h.nbl_ok, erec_ok = h.erec_ok;
      qual_ready = h.qual_ready, cells_clean = h.cells_clean, par = h.par, n = h.n, m = h.m;
      n_sorted = h.n_sorted, n_flagged = h.n_flagged, cells_nkeys = h.cells_nkeys;
      skeys = h.skeys, svals = h.svals, cells_keys = h.cells_keys;
      if (e == hipSuccess) e = hipGraphInstantiateWithFlags(&g->exec, rec, 0);
      if (rec) (void)hipGraphDestroy(rec);
      if (e != hipSuccess) {
        g->exec = nullptr;
        graphs_work = false;
        (void)hipGetLastError();
        return false;
      }
    }
    if (hipGraphLaunch(g->exec, st) != hipSuccess) {
      graphs_work = false;
      (void)hipGetLastError();
      return false;
    }
    rep_want++;
    // the host's state after q_step
    std::swap(cur, alt);
    flipped = !flipped;
    par ^= 1;
    skeys = sc.keys_alt;
    svals = sc.vals_alt;
    n_sorted = n;
    cells_keys = nullptr;
    cells_clean = false;
    nbl_ok = false;
    erec_ok = !(flags & (SPH_STEP_SPLIT | SPH_STEP_MERGE));
    if (flags & SPH_STEP_SPLIT) n_flagged = n;
    return true;
  }

  void clear_force_flags() {
    // force_waiting* and the 2D mouse force last one step (SPH-3D-2/sph_system.cpp:403)
    if (variant == SPH_V2D) ((SphSysParam2D *)raw)->force_waiting = false;
    else {
      ((SphSysParam3D *)raw)->flag0 = false;
      if (variant == SPH_V3D4) ((SphSysParam3D *)raw)->flag1 = false;
    }
    P.push_left = P.push_right = 0;
    P.mouse = 0;
  }
};

#define CHECK_CTX(c)            \
  do {                          \
    if (!(c)) return SPH_EINVAL; \
  } while (0)

extern "C" {

const char *sph_version(void) { return SPH_VERSION; }

int sph_param_defaults(int variant, void *out) {
  if (!valid_variant(variant) || !out) return SPH_EINVAL;
  if (variant == SPH_V2D) defaults2(*(SphSysParam2D *)out);
  else defaults3(variant, *(SphSysParam3D *)out);
  return SPH_OK;
}

int sph_param_derive(int variant, void *inout) {
  if (!valid_variant(variant) || !inout) return SPH_EINVAL;
  if (variant == SPH_V2D) {
    SphSysParam2D &s = *(SphSysParam2D *)inout;
    if (!(s.large_kernel > 0.0f) || !(s.small_kernel > 0.0f)) return SPH_EINVAL;
    derive2(s);
  } else {
    SphSysParam3D &s = *(SphSysParam3D *)inout;
    if (!(s.large_kernel > 0.0f) || !(s.small_kernel > 0.0f)) return SPH_EINVAL;
    derive3(s);
  }
  return SPH_OK;
}

int sph_ctx_create(int variant, const void *sysparam, uint32_t capacity, uint32_t max_triangles,
                   SphCtx **out) {
  if (!out) return SPH_EINVAL;
  *out = nullptr;
  // particle indices share a 32-bit word with a 5-bit cell-offset id in the pair lists
  if (!valid_variant(variant) || !sysparam || capacity == 0 || capacity > (1u << 27)) return SPH_EINVAL;
  SphCtx *c = new (std::nothrow) SphCtx();
  if (!c) return SPH_ECAP;
  c->variant = variant;
  c->raw_size = variant == SPH_V2D ? sizeof(SphSysParam2D) : sizeof(SphSysParam3D);
  std::memcpy(c->raw, sysparam, c->raw_size);
  c->cap = capacity;
  c->max_tri = max_triangles;
  c->P = make_dev_params(variant, c->raw, capacity);
  if (c->P.total_cell == 0) {
    delete c;
    return SPH_EINVAL;
  }
  c->kbits = key_bits(c->P.total_cell);
  c->dgrid_cells = dgrid_cell_blocks_exact(c->P);
  if (hipStreamCreateWithFlags(&c->st, hipStreamNonBlocking) != hipSuccess) {
    delete c;
    return SPH_EHIP;
  }
  const size_t cap = capacity;
  bool ok = c->alloc_state(c->cur) && c->alloc_state(c->alt) && c->alloc(c->keys, cap) &&
            c->alloc(c->vals, cap) && c->alloc(c->sc.keys_alt, cap) && c->alloc(c->sc.vals_alt, cap) &&
            c->alloc(c->sc.tile_hist, sph_sort_hist_elems(cap)) &&
            c->alloc(c->s2p_hash, cap) && c->alloc(c->s2p_cell, cap) &&
            c->alloc(c->cstart, c->P.total_cell) && c->alloc(c->cend, c->P.total_cell) &&
            c->alloc(c->sb.split, sph_bit_words(cap)) && c->alloc(c->sb.dead, sph_bit_words(cap)) &&
            c->alloc(c->sb.qual, sph_bit_words(cap)) && c->alloc(c->sb.toff, sph_bit_tiles(cap)) &&
            c->alloc(c->newslot, cap) && c->alloc(c->q2d, std::max<size_t>(c->P.total_cell, 1)) &&
            c->alloc(c->cnt, 1) && c->alloc(c->rep_seq, 1) && c->alloc(c->aos_dev, cap * sizeof(SphParticle3D)) &&
            c->alloc(c->aux.frec, 3 * (size_t)cap) && c->alloc(c->aux.erec, cap) && c->alloc(c->aux.ez, cap) && c->alloc(c->aux.qpos, cap) &&
            c->alloc(c->aux.nbl, (size_t)SPH_NBL_K * cap) && c->alloc(c->aux.nbl_cnt, cap);
  c->aux.nbl_stride = cap;
  if (ok && c->P.dim == 3 && c->P.tot_dens > 0) {
    c->ncube = mc_segments(c->P);
    ok = c->alloc(c->dgrid, c->P.tot_dens) && c->alloc(c->normal3, (size_t)c->P.tot_dens * 3) &&
         c->alloc(c->cube_count, c->ncube) && c->alloc(c->cube_off, c->ncube) &&
         c->alloc(c->seg_cube, c->ncube) && c->alloc(c->seg_coff, c->ncube) &&
         c->alloc(c->clist, (size_t)std::max<uint32_t>(max_triangles, 1)) &&
         c->alloc(c->tris, (size_t)std::max<uint32_t>(max_triangles, 1) * 18);
    if (ok) ok = c->alloc(c->occ, 2 * sph_occ_words(c->P.total_cell));
  }
  size_t scan_elems = sph_scan_tmp_elems(std::max(cap, c->ncube));
  ok = ok && c->alloc(c->scan_tmp, scan_elems);
  c->sb.scan_tmp = c->scan_tmp;
  if (ok && sph_use_bins(c->P.total_cell, cap)) {
    c->bins.hkey = c->keys;
    c->bins.rank = c->vals;
    c->bins.bslot = c->s2p_hash;
    ok = c->alloc(c->bins.ccount, c->P.total_cell) &&
         c->alloc(c->bins.tmp, sph_bin_tiles(c->P.total_cell));
    if (ok) sph_fill_u32(c->bins.ccount, 0u, c->P.total_cell, c->st);
  }
  if (ok && (hipHostMalloc((void **)&c->rep, sizeof(Report), hipHostMallocDefault) != hipSuccess ||
             hipHostGetDevicePointer((void **)&c->rep_dev, c->rep, 0) != hipSuccess))
    ok = false;
  if (ok && !c->tune.create()) ok = false;
  c->tune.start(kTuneRounds, kTuneAfter, kTuneEvery);
  if (!ok) {
    delete c;
    return SPH_ECAP;
  }
  std::memset(c->rep, 0, sizeof(Report));
  sph_fill_u32(c->rep_seq, 0u, 1, c->st);
  launch_upload(variant, c->aos_dev, 0, c->cur, 0, c->st, c->cnt, 0, 0);
  if (c->sync() != SPH_OK) {
    delete c;
    return SPH_EHIP;
  }
  *out = c;
  return SPH_OK;
}

int sph_ctx_destroy(SphCtx *ctx) {
  CHECK_CTX(ctx);
  delete ctx;
  return SPH_OK;
}

int sph_set_params(SphCtx *ctx, const void *sysparam) {
  CHECK_CTX(ctx);
  if (!sysparam) return SPH_EINVAL;
  DevParams P = make_dev_params(ctx->variant, sysparam, ctx->cap);
  if (P.total_cell != ctx->P.total_cell || P.tot_dens != ctx->P.tot_dens) return SPH_EINVAL;
  std::memcpy(ctx->raw, sysparam, ctx->raw_size);
  if (std::memcmp(&P, &ctx->P, sizeof(P)) != 0) ctx->drop_graphs();  // they hold the parameters
  ctx->P = P;
  ctx->nbl_ok = false;   // the pair lists were made with the old kernel radii
  ctx->erec_ok = false;  // and the quantised positions with the old steps and marks
  return SPH_OK;
}

int sph_get_params(SphCtx *ctx, void *out) {
  CHECK_CTX(ctx);
  if (!out) return SPH_EINVAL;
  std::memcpy(out, ctx->raw, ctx->raw_size);
  return SPH_OK;
}

int sph_upload_particles(SphCtx *ctx, const void *aos, uint32_t n) {
  CHECK_CTX(ctx);
  if (n > ctx->cap) return SPH_ECAP;
  if (n > 0 && !aos) return SPH_EINVAL;
  const size_t rec = ctx->variant == SPH_V2D ? sizeof(SphParticle2D) : sizeof(SphParticle3D);
  if (n > 0 && hipMemcpyAsync(ctx->aos_dev, aos, rec * n, hipMemcpyHostToDevice, ctx->st) != hipSuccess)
    return SPH_EHIP;
  launch_upload(ctx->variant, ctx->aos_dev, n, ctx->cur, 0, ctx->st, ctx->cnt, n, n);
  ctx->hashed = ctx->sorted = ctx->lists_valid = ctx->merged = false;
  ctx->erec_ok = false;
  ctx->nbl_ok = false;
  return ctx->sync();
}

int sph_download_particles(SphCtx *ctx, void *aos, uint32_t n) {
  CHECK_CTX(ctx);
  if (n > ctx->n) return SPH_EINVAL;
  if (n == 0) return SPH_OK;
  if (!aos) return SPH_EINVAL;
  const size_t rec = ctx->variant == SPH_V2D ? sizeof(SphParticle2D) : sizeof(SphParticle3D);
  launch_download(ctx->variant, ctx->cur, Span{0u, ctx->m, 0u, 0u}, n, ctx->aos_dev, ctx->st);
  if (hipMemcpyAsync(aos, ctx->aos_dev, rec * n, hipMemcpyDeviceToHost, ctx->st) != hipSuccess)
    return SPH_EHIP;
  return ctx->drain();
}

int sph_num_particles(SphCtx *ctx, uint32_t *n) {
  CHECK_CTX(ctx);
  if (!n) return SPH_EINVAL;
  *n = ctx->n;
  return SPH_OK;
}

int sph_calc_hash(SphCtx *ctx) {
  CHECK_CTX(ctx);
  if (ctx->n == 0) return SPH_OK;
  ctx->q_hash();
  int rc = ctx->sync();
  if (rc) return rc;
  ctx->hashed = true;
  ctx->sorted = ctx->lists_valid = ctx->merged = false;
  return ctx->rep->c.err ? SPH_EDOMAIN : SPH_OK;
}

int sph_sort(SphCtx *ctx) {
  CHECK_CTX(ctx);
  if (ctx->n == 0) return SPH_OK;
  if (!ctx->hashed) return SPH_EINVAL;
  ctx->q_sort();
  int rc = ctx->sync();
  if (rc) return rc;
  ctx->sorted = true;
  return SPH_OK;
}

int sph_cell_ranges(SphCtx *ctx) {
  CHECK_CTX(ctx);
  if (ctx->n == 0) return SPH_OK;
  if (!ctx->sorted) return SPH_EINVAL;
  ctx->q_cells();
  int rc = ctx->sync();
  if (rc) return rc;
  ctx->lists_valid = true;
  ctx->hashed = false;
  return SPH_OK;
}

#define PHASE_BODY(ctx, need_lists, call)            \
  CHECK_CTX(ctx);                                    \
  if ((ctx)->n == 0) return SPH_EEMPTY;              \
  if ((need_lists) && !(ctx)->lists_valid) return SPH_EINVAL; \
  if ((ctx)->m != (ctx)->n) return SPH_EINVAL;       \
  (ctx)->call;                                       \
  return (ctx)->sync();

int sph_density(SphCtx *ctx) { PHASE_BODY(ctx, true, q_density()) }
int sph_force(SphCtx *ctx) { PHASE_BODY(ctx, true, q_force()) }
int sph_energy(SphCtx *ctx) { PHASE_BODY(ctx, true, q_energy()) }

int sph_integrate(SphCtx *ctx) {
  CHECK_CTX(ctx);
  if (ctx->n == 0) return SPH_OK;
  if (ctx->m != ctx->n) return SPH_EINVAL;
  ctx->q_integrate();
  return ctx->sync();
}

int sph_split(SphCtx *ctx, uint32_t *n_requested, uint32_t *n_done) {
  CHECK_CTX(ctx);
  if (n_requested) *n_requested = 0;
  if (n_done) *n_done = 0;
  if (ctx->n == 0) return SPH_OK;
  if (ctx->m != ctx->n) return SPH_EINVAL;
  launch_begin_step(ctx->cnt, ctx->st);  // resets split/merge counters, n_pre = n
  ctx->q_split();
  int rc = ctx->sync();
  if (rc) return rc;
  if (n_requested) *n_requested = ctx->rep->c.s_req;
  if (n_done) *n_done = ctx->rep->c.s_done;
  return SPH_OK;
}

int sph_merge(SphCtx *ctx, uint32_t *groups) {
  CHECK_CTX(ctx);
  if (groups) *groups = 0;
  if (!ctx->lists_valid) return SPH_EINVAL;
  ctx->q_merge();
  int rc = ctx->sync();
  if (rc) return rc;
  ctx->merged = true;
  if (groups) *groups = ctx->rep->c.groups;
  return SPH_OK;
}

int sph_compact(SphCtx *ctx, uint32_t *n_out) {
  CHECK_CTX(ctx);
  if (!ctx->merged) return SPH_EINVAL;
  ctx->q_compact();
  int rc = ctx->sync();
  if (rc) return rc;
  ctx->merged = false;
  ctx->lists_valid = false;
  ctx->compacted = true;
  ctx->n_status = ctx->m;
  if (n_out) *n_out = ctx->n;
  return SPH_OK;
}

int sph_density_grid(SphCtx *ctx) {
  CHECK_CTX(ctx);
  if (ctx->P.dim != 3 || !ctx->dgrid) return SPH_EINVAL;
  if (!ctx->lists_valid) return SPH_EINVAL;
  ctx->q_dgrid();
  return ctx->sync();
}

int sph_grid_normals(SphCtx *ctx) {
  CHECK_CTX(ctx);
  if (ctx->P.dim != 3 || !ctx->dgrid) return SPH_EINVAL;
  ctx->q_normals();
  return ctx->sync();
}

int sph_marching_cubes(SphCtx *ctx, uint32_t *n_tri) {
  CHECK_CTX(ctx);
  if (ctx->P.dim != 3 || !ctx->dgrid) return SPH_EINVAL;
  ctx->q_mc();
  int rc = ctx->sync();
  if (rc) return rc;
  if (n_tri) *n_tri = ctx->rep->c.ntri;
  return ctx->rep->c.ntri > ctx->max_tri ? SPH_ETRI : SPH_OK;
}

int sph_step(SphCtx *ctx, uint32_t flags, uint32_t *n_out) {
  CHECK_CTX(ctx);
  if (ctx->n == 0) return SPH_EEMPTY;
  ctx->aux.choose_forms(ctx->variant, false, ctx->n);
  ctx->tune.force_counts = !ctx->aux.fine_force;
  const bool reported = ctx->graph_step(flags);
  if (!reported) ctx->q_step(flags);
  // the cell-range phase made physical == live before split appended children
  int rc = ctx->sync(reported);
  if (rc == SPH_OK) ctx->tune.end_step();
  ctx->clear_force_flags();
  ctx->hashed = ctx->sorted = ctx->merged = false;
  ctx->lists_valid = !(flags & SPH_STEP_MERGE);
  if (rc) return rc;
  if (flags & SPH_STEP_MERGE) ctx->n_status = ctx->m;
  if (n_out) *n_out = ctx->n;
  return ctx->rep->c.err ? SPH_EDOMAIN : SPH_OK;
}

static size_t count_of(SphCtx *ctx, int which) {
  switch (which) {
    case SPH_Q_HASH:
    case SPH_Q_INDEX: return ctx->skeys ? ctx->n_sorted : 0;
    case SPH_Q_START:
    case SPH_Q_END: return ctx->P.total_cell;
    case SPH_Q_SPLITFLAG: return ctx->n_flagged;
    case SPH_Q_STATUS: return ctx->n_status;
    case SPH_Q_COUNTERS: return sizeof(Counters) / 4;
    case SPH_Q_DGRID: return ctx->dgrid ? ctx->P.tot_dens : 0;
    case SPH_Q_NORMAL: return ctx->dgrid ? (size_t)ctx->P.tot_dens * 3 : 0;
    case SPH_Q_TRI: {
      uint nt = ctx->rep->c.ntri < ctx->max_tri ? ctx->rep->c.ntri : ctx->max_tri;
      return ctx->tris ? (size_t)nt * 18 : 0;
    }
  }
  return 0;
}

int sph_count(SphCtx *ctx, int which, size_t *n) {
  CHECK_CTX(ctx);
  if (!n) return SPH_EINVAL;
  *n = count_of(ctx, which);
  return SPH_OK;
}

// Reads an integer array; SPLITFLAG and STATUS use the reference's conventions
// (dev_split: 0 = split; dev_status: 1 = removed), indexed by slot.
int sph_get_u32(SphCtx *ctx, int which, uint32_t *out, size_t n) {
  CHECK_CTX(ctx);
  if (n == 0) return SPH_OK;
  if (!out || n > count_of(ctx, which)) return SPH_EINVAL;
  const uint *src = nullptr;
  switch (which) {
    case SPH_Q_HASH: src = ctx->skeys; break;
    case SPH_Q_INDEX: src = ctx->svals; break;
    case SPH_Q_START: src = ctx->cstart; break;
    case SPH_Q_END: src = ctx->cend; break;
    case SPH_Q_SPLITFLAG: src = ctx->sb.split; break;
    case SPH_Q_STATUS: src = ctx->sb.dead; break;
    case SPH_Q_COUNTERS: src = (const uint *)ctx->cnt; break;
    default: return SPH_EINVAL;
  }
  // bits arrive in the first words of out and are spread from the last entry down (word k / 32 is
  // still there when entry k is written)
  const bool bits = which == SPH_Q_SPLITFLAG || which == SPH_Q_STATUS;
  if (hipMemcpyAsync(out, src, (bits ? (n + 31) / 32 : n) * 4, hipMemcpyDeviceToHost, ctx->st) != hipSuccess)
    return SPH_EHIP;
  int rc = ctx->drain();
  if (rc) return rc;
  for (size_t k = bits ? n : 0; k-- > 0;)
    out[k] = ((out[k >> 5] >> (k & 31)) & 1u) ^ (which == SPH_Q_SPLITFLAG ? 1u : 0u);
  return SPH_OK;
}

int sph_get_f32(SphCtx *ctx, int which, float *out, size_t n) {
  CHECK_CTX(ctx);
  if (n == 0) return SPH_OK;
  if (!out || n > count_of(ctx, which)) return SPH_EINVAL;
  const float *src = nullptr;
  switch (which) {
    case SPH_Q_DGRID: src = ctx->dgrid; break;
    case SPH_Q_NORMAL: src = ctx->normal3; break;
    case SPH_Q_TRI: src = ctx->tris; break;
    default: return SPH_EINVAL;
  }
  if (hipMemcpyAsync(out, src, n * 4, hipMemcpyDeviceToHost, ctx->st) != hipSuccess) return SPH_EHIP;
  return ctx->drain();
}

int sph_autotune(SphCtx *ctx, uint32_t rounds, uint32_t after_steps, uint32_t every_steps) {
  CHECK_CTX(ctx);
  ctx->tune.start(rounds, after_steps, every_steps);
  return SPH_OK;
}

int sph_set_lists(SphCtx *ctx, uint32_t force_list, uint32_t energy_list) {
  CHECK_CTX(ctx);
  return ctx->tune.set(force_list, energy_list) ? SPH_OK : SPH_EINVAL;
}

int sph_tuned_lists(SphCtx *ctx, uint32_t *force_list, uint32_t *energy_list, float *best_ms) {
  CHECK_CTX(ctx);
  if (force_list) *force_list = (uint32_t)kForceLists[ctx->tune.force];
  if (energy_list) *energy_list = (uint32_t)kEnergyLists[ctx->tune.energy];
  if (best_ms)
    for (int k = 0; k < 2; k++)
      for (int c = 0; c < 3; c++) best_ms[k * 3 + c] = ctx->tune.best[k][c];
  return SPH_OK;
}

int sph_prof_enable(SphCtx *ctx, int on) {
  CHECK_CTX(ctx);
  ctx->prof_mask = on ? (1u << SPH_P_COUNT) - 1u : 0u;
  return SPH_OK;
}

int sph_prof_phases(SphCtx *ctx, uint32_t phase_mask) {
  CHECK_CTX(ctx);
  ctx->prof_mask = phase_mask & ((1u << SPH_P_COUNT) - 1u);
  return SPH_OK;
}

int sph_prof_reset(SphCtx *ctx) {
  CHECK_CTX(ctx);
  int rc = ctx->sync();
  for (int k = 0; k < SPH_P_COUNT; k++) {
    ctx->prof_ms[k] = 0.0;
    ctx->prof_n[k] = 0;
  }
  return rc;
}

int sph_prof_read(SphCtx *ctx, int phase, double *ms_total, uint64_t *launches) {
  CHECK_CTX(ctx);
  if (phase < 0 || phase >= SPH_P_COUNT) return SPH_EINVAL;
  if (ms_total) *ms_total = ctx->prof_ms[phase];
  if (launches) *launches = ctx->prof_n[phase];
  return SPH_OK;
}

int sph_synchronize(SphCtx *ctx) {
  CHECK_CTX(ctx);
  return ctx->sync();
}

}  // extern "C"
