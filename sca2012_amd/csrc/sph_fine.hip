// Neighbour kernels with several lanes per particle (density, force, energy), for scenes that
// do not fill the GPU with one thread per particle (sph_kernels.hip has that form). There, a
// thread walks its particle's 27 cells one after another and the launch takes as long as that
// chain of dependent loads, whatever the particle count; here the chain is split:
//   density, energy  nine lanes per particle, seven particles per wave. In 3D a lane takes one
//                    row of three cells along x, which is one contiguous run of the sorted
//                    particles; in 2D it takes one cell.
//   force            eight lanes per particle, each evaluating every eighth pair of its list.
// Sums keep the reference's order: a cell's partial belongs to one lane, the 27 partials are
// added in offset order, and values summed pair by pair are computed in parallel, exchanged
// through LDS and added by one lane per component, in list order. So every result has the
// bits of the one-thread-per-particle kernels. Exchanges stay within a wave, so no block
// barrier is needed.
#include "sph_device.h"

namespace {

constexpr int FL = 9;               // lanes of a particle in the density and energy kernels
constexpr int FP = 64 / FL;         // particles of a wave (lane 63 idles: row FP of the LDS arrays)
constexpr int FB = FP * (BLK / 64);  // particles of a block

// LDS written by some lanes of the wave is read by others after this
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The cells a lane walks: the run [s, e) of sorted particles, its cells [s, b1), [b1, b2) and
// [b2, e) at offset indices o[0..2] (2D: one cell, b1 = b2 = e).
struct Row {
  uint s, e, b1, b2;
  int o[3];
  __device__ int cell(uint j) const { return j < b1 ? 0 : (j < b2 ? 1 : 2); }
};

template <int V>
__device__ inline Row load_row(const DevParams &P, int r, const uint c[3], bool valid,
                               const uint *__restrict__ cstart, const uint *__restrict__ cend) {
  Row R;
  if constexpr (VT<V>::dim == 3) {
    // offset indices (SPH-3D-2/sph_system.cu:456-562) of dx = -1, 0, 1 in row dy of a layer
    constexpr uint kRow[3] = {1u | 3u << 8 | 7u << 16, 2u | 0u << 8 | 5u << 16, 8u | 6u << 8 | 4u << 16};
    const int dy = r % 3 - 1, dz = r / 3 - 1;
    const int layer = dz == 0 ? 0 : (dz < 0 ? 9 : 18);
    const uint code = dy < 0 ? kRow[0] : (dy == 0 ? kRow[1] : kRow[2]);
#pragma unroll
    for (int k = 0; k < 3; k++) R.o[k] = layer + (int)((code >> (8 * k)) & 0xffu);
    const uint y = c[1] + (uint)dy, z = c[2] + (uint)dz;  // -1 wraps and fails the test
    const bool ok = valid && y < P.ncell[1] && z < P.ncell[2];
    const uint h = P.cell_base + (z * P.ncell[1] + y) * P.ncell[0] + c[0];
    const bool ok0 = ok && c[0] > 0u, ok2 = ok && c[0] + 1u < P.ncell[0];
    const uint s0 = ok0 ? cstart[h - 1] : SPH_EMPTY, s1 = ok ? cstart[h] : SPH_EMPTY,
               s2 = ok2 ? cstart[h + 1] : SPH_EMPTY;
    const uint e0 = ok0 ? cend[h - 1] : 0u, e1 = ok ? cend[h] : 0u, e2 = ok2 ? cend[h + 1] : 0u;
    R.s = min(s0, min(s1, s2));  // starts ascend; an empty cell holds SPH_EMPTY and 0
    R.e = max(e0, max(e1, e2));
    if (R.s == SPH_EMPTY) R.s = R.e = 0u;
    R.b1 = s0 != SPH_EMPTY ? e0 : R.s;
    R.b2 = s1 != SPH_EMPTY ? e1 : R.b1;
  } else {
    R.o[0] = R.o[1] = R.o[2] = r;
    R.s = R.e = 0u;
    if (valid) nb_range<V>(P, r, c, cstart, cend, R.s, R.e);
    R.b1 = R.b2 = R.e;
  }
  return R;
}

__device__ inline unsigned long long low_bits(uint n) {
  return n >= 64u ? ~0ull : (1ull << n) - 1ull;
}

// Bit k = test(entry s + k) over a run of at most 64, eight positions in flight.
template <class T>
__device__ inline unsigned long long run_mask(const __amdgpu_buffer_rsrc_t prs, uint s, uint e,
                                              T &&test) {
  unsigned long long m = 0ull;
  for (uint j = s; j < e; j += 8) {
    float4 q[8];
    sph_group4(prs, j, q);
    sph_group4(prs, j + 4, q + 4);
    uint b = 0;
#pragma unroll
    for (int k = 0; k < 8; k++) b |= test(q[k]) ? 1u << k : 0u;
    m |= (unsigned long long)b << (j - s);
  }
  return m & low_bits(e - s);
}

// f(j, position of j) for the entries of a mask over [s, s + 64), in order, the next
// position requested before f runs on the one before it
template <class F>
__device__ inline void each_bit(const float4 *__restrict__ pos, uint s, unsigned long long m, F &&f) {
  if (!m) return;
  uint j = s + (uint)__builtin_ctzll(m);
  float4 p = pos[j];
  for (;;) {
    m &= m - 1ull;
    const uint jn = m ? s + (uint)__builtin_ctzll(m) : j;
    const float4 pn = pos[jn];
    f(j, p);
    if (!m) break;
    j = jn;
    p = pn;
  }
}

// Exclusive prefix, in offset order, of the counts that the lanes of each particle hold for
// their cells; tot = their sum. `row` is the particle's 28 words of LDS.
template <bool D3>
__device__ inline void cell_prefix(uint *row, int r, const Row &R, const uint n[3], uint b[3], uint &tot) {
  const int lane = threadIdx.x & 63;
  uint a0 = n[0], a1 = 0, a2 = 0;
  if (D3) {
#pragma unroll
    for (int k = 0; k < 3; k++) row[R.o[k]] = n[k];
    wave_sync();
    a0 = row[3 * r], a1 = row[3 * r + 1], a2 = row[3 * r + 2];
  }
  uint x = a0 + a1 + a2;
  const uint own = x;
#pragma unroll
  for (int d = 1; d < FL; d <<= 1) {
    const uint y = __shfl_up(x, d, 64);
    if (r >= d) x += y;
  }
  tot = __shfl(x, min(lane - r + FL - 1, 63), 64);
  const uint ex = x - own;
  if (D3) {
    wave_sync();
    row[3 * r] = ex;
    row[3 * r + 1] = ex + a0;
    row[3 * r + 2] = ex + a0 + a1;
    wave_sync();
#pragma unroll
    for (int k = 0; k < 3; k++) b[k] = row[R.o[k]];
    wave_sync();
  } else {
    b[0] = b[1] = b[2] = ex;
  }
}

// ---------------------------------------------------------------------------------------
// Density, pressure, the force pair list and the force kernel's record: k_density
// (sph_kernels.hip) in nine lanes per particle.
// ---------------------------------------------------------------------------------------
template <int V, bool B>
__global__ __launch_bounds__(BLK) void k_density_fine(
    DevParams P0, const DevParams *__restrict__ Ptab, const uint *__restrict__ slot,
    const float4 *__restrict__ pos, const float4 *__restrict__ ev, float2 *__restrict__ dp,
    float *__restrict__ frec, const uint *__restrict__ cstart, const uint *__restrict__ cend,
    const uint *n_dev, uint n_host, uint *__restrict__ nbl, uint *__restrict__ nbl_cnt,
    uint nbl_stride) {
  constexpr bool D3 = VT<V>::dim == 3;
  __shared__ __align__(16) uint sh[BLK / 64][FP + 1][28];
  const uint n = dev_count(n_dev, n_host);
  const uint nvb = (n + FB - 1) / FB;
  if (blockIdx.x >= nvb) return;
  const uint wave = threadIdx.x >> 6;
  const int lane = (int)(threadIdx.x & 63u), q = lane / FL, r = lane % FL;
  const uint i = xcd_block(blockIdx.x, nvb) * FB + wave * FP + (uint)q;
  const bool act = q < FP && i < n;
  uint *const row = sh[wave][q];
  const uint ic = act ? i : 0u;
  const __amdgpu_buffer_rsrc_t prs = sph_rsrc(pos, n_host);
  const DevParams &P = scene_params<B>(P0, Ptab, B ? slot[ic] : 0u);
  const float4 pi = pos[ic];
  const int L = lvl_index(pi.w);
  const float k2 = L ? P.k2[1] : P.k2[0];
  const float k6 = L ? P.k6[1] : P.k6[0];
  const float poly6 = L ? P.poly6[1] : P.poly6[0];
  const float mi = L ? P.mass[1] : P.mass[0];
  const float eps = P.dens_eps, feps = D3 ? eps : 0.0001f;
  const float mp0 = P.mass[0] * poly6, mp1 = P.mass[1] * poly6;
  const float self_t = mi * poly6 * k6;
  const float fk0 = k2 > P.k2[0] ? k2 : P.k2[0], fk1 = k2 > P.k2[1] ? k2 : P.k2[1];
  uint c[3];
  const bool valid = cell_of<V>(P, pi.x, pi.y, pi.z, c);
  const Row R = load_row<V>(P, r, c, act && valid, cstart, cend);
  auto dist2 = [&](const float4 &pj) {
    const float dx = pj.x - pi.x, dy = pj.y - pi.y;
    if (D3) {
      const float dz = pj.z - pi.z;
      return dx * dx + dy * dy + dz * dz;
    }
    return dx * dx + dy * dy;
  };
  // listed: the force kernel's pairs; near: those and (2D) the closer pairs that only the
  // density sums. The particle itself is summed, and listed in 2D only.
  auto listed = [&](const float4 &pj, float r2) {
    return !(r2 < feps) && r2 < (lvl_index(pj.w) ? fk1 : fk0);
  };
  auto near = [&](const float4 &pj, float r2) {
    return !(r2 < eps) && r2 < (lvl_index(pj.w) ? fk1 : fk0);
  };
  const bool self_here = i >= R.s && i < R.e;
  const bool wide = __any(R.e - R.s > 64u);  // some run does not fit a 64-bit mask
  unsigned long long m = 0ull;
  uint cn[3] = {0u, 0u, 0u}, base[3], nc;
  if (!wide) {
    m = run_mask(prs, R.s, R.e, [&](const float4 &pj) { return near(pj, dist2(pj)); });
    unsigned long long ml = m;
    if (!D3)
      ml = run_mask(prs, R.s, R.e, [&](const float4 &pj) { return listed(pj, dist2(pj)); });
    if (self_here) {
      m |= 1ull << (i - R.s);
      if (!D3) ml |= 1ull << (i - R.s);
    }
    const unsigned long long l1 = low_bits(R.b1 - R.s), l2 = low_bits(R.b2 - R.s);
    cn[0] = (uint)__popcll(ml & l1);
    cn[1] = (uint)__popcll(ml & l2 & ~l1);
    cn[2] = (uint)__popcll(ml & ~l2);
  } else {
    for (uint j = R.s; j < R.e; j++) {
      const float4 pj = pos[j];
      const bool h = (!D3 && j == i) || listed(pj, dist2(pj));
      const int k = R.cell(j);
#pragma unroll
      for (int t = 0; t < 3; t++) cn[t] += (h && k == t) ? 1u : 0u;
    }
  }
  cell_prefix<D3>(row, r, R, cn, base, nc);
  float cs[3] = {0.0f, 0.0f, 0.0f};
  uint *const my = nbl ? nbl + 4 * (size_t)ic : nullptr;  // entry e at (e / 4) 4 nbl_stride + e mod 4
  const size_t gs = 4 * (size_t)nbl_stride;
  auto hit = [&](uint j, const float4 &pj) {
    const float r2 = dist2(pj);
    const float d = k2 - r2;
    const float tv = (lvl_index(pj.w) ? mp1 : mp0) * ((d * d) * d);
    const float t = (!(r2 < eps) && r2 < k2) ? tv : (j == i ? self_t : 0.0f);
    const int k = R.cell(j);
    const bool in_list = D3 ? j != i : (j == i || !(r2 < feps));
#pragma unroll
    for (int x = 0; x < 3; x++)
      if (k == x) {
        cs[x] = cs[x] + t;
        if (my && in_list) {
          if (base[x] < SPH_NBL_K) my[(base[x] >> 2) * gs + (base[x] & 3u)] = pack_entry(R.o[x], j);
          base[x]++;
        }
      }
  };
  if (!wide) {
    each_bit(pos, R.s, m, hit);
  } else {
    for (uint j = R.s; j < R.e; j++) {
      const float4 pj = pos[j];
      if (j == i || near(pj, dist2(pj))) hit(j, pj);
    }
  }
  // the cells' partials, added in offset order by every lane of the particle
  float *const frow = reinterpret_cast<float *>(row);
#pragma unroll
  for (int k = 0; k < (D3 ? 3 : 1); k++) frow[R.o[k]] = cs[k];
  wave_sync();
  float total = 0.0f;
#pragma unroll
  for (int o = 0; o < VT<V>::nnb; o++) total = total + frow[o];
  if (!act) return;
  const float qd = total / P.rest_density;
  const float press = ((qd * qd) * qd - 1.0f) * P.gas_constant;
  if (r == 0 && nbl) nbl_cnt[i] = nc;
  // the record's quotients (layout at struct Aux), one per lane:
  //   m/dens, press/dens^2, ((-1*grad_L)*m)/dens for L = 0, 1, (lapc_L*m)/dens for L = 0, 1
  const float den = r == 1 ? total * total : total;
  float num = r == 0 ? mi : press;
  if (D3) {
    const float g = (-1.0f) * (r == 2 ? P.grad[0] : P.grad[1]) * mi;
    const float l = (r == 4 ? P.lapc[0] : P.lapc[1]) * mi;
    num = r < 2 ? num : (r < 4 ? g : l);
  }
  const float v = num / den;
  float *const rec = frec + 12 * (size_t)i;
  const float4 evi = ev[i];
  if (r < 2) {
    rec[r] = v;
  } else if (r < 6) {
    if (D3) rec[r == 2 ? 4 : (r == 3 ? 8 : (r == 4 ? 5 : 9))] = v;
  } else if (r == 6) {
    *reinterpret_cast<float2 *>(rec + 2) = make_float2(evi.x, evi.y);
  } else if (r == 7) {
    if (D3) *reinterpret_cast<float2 *>(rec + 6) = make_float2(evi.z, 0.0f);
    dp[i] = make_float2(total, press);
  } else if (D3) {
    *reinterpret_cast<float2 *>(rec + 10) = make_float2(evi.z, 0.0f);
  }
}

// ---------------------------------------------------------------------------------------
// Force: k_force (sph_kernels.hip) in eight lanes per particle. A round evaluates up to eight
// pairs of each particle, one per lane, and exchanges their contributions through LDS; lane
// c < 7 then adds component c (force x, y, z; colour gradient x, y, z; colour laplacian) of the
// eight pairs in order. Adding the +0 of a pair that does not contribute changes no bits: a
// running sum starts at +0 and so is never -0.
// ---------------------------------------------------------------------------------------
constexpr int GL = 8;                // lanes of a particle
constexpr int GB = BLK / GL;         // particles of a block
constexpr int GC = 20;               // words per component: 8 (a, b) pairs, padded against conflicts
constexpr int GQ = 16;               // entries of the walk's queue

template <int V, bool B>
__global__ __launch_bounds__(BLK) void k_force_fine(
    DevParams P0, const DevParams *__restrict__ Ptab, const uint *__restrict__ slot,
    const float4 *__restrict__ pos, const float4 *__restrict__ ev, const float2 *__restrict__ dp,
    const float4 *__restrict__ frec, float *__restrict__ acc, const uint *__restrict__ cstart,
    const uint *__restrict__ cend, const uint *n_dev, uint n_host, const uint *__restrict__ nbl,
    const uint *__restrict__ nbl_cnt, uint nbl_stride) {
  constexpr bool D3 = VT<V>::dim == 3;
  __shared__ __align__(16) float sh[GB][7][GC];
  __shared__ uint queue[GB][GQ];
  const uint n = dev_count(n_dev, n_host);
  const uint nvb = (n + GB - 1) / GB;
  if (blockIdx.x >= nvb) return;
  const uint g = threadIdx.x / GL;
  const int l = (int)(threadIdx.x % GL), lane = (int)(threadIdx.x & 63u), g0 = lane - l;
  const uint i = xcd_block(blockIdx.x, nvb) * GB + g;
  const bool act = i < n;
  const uint ic = act ? i : 0u;
  const DevParams &P = scene_params<B>(P0, Ptab, B ? slot[ic] : 0u);
  const float4 pi = pos[ic];
  const float4 evi = ev[ic];
  const float4 fri = frec[3 * (size_t)ic];
  const int Li = lvl_index(pi.w);
  const float hi = Li ? P.kernel[1] : P.kernel[0];
  const float mi = Li ? P.mass[1] : P.mass[0];
  const float k2i = Li ? P.k2[1] : P.k2[0];
  const float spi = Li ? P.spiky[1] : P.spiky[0];
  const float k6i = Li ? P.k6[1] : P.k6[0];
  const float rk6i = Li ? P.rcp_k6[1] : P.rcp_k6[0];
  const bool k6_fast = P.k6_fast != 0;
  const float vki = Li ? P.visco_k6[1] : P.visco_k6[0];
  const float gi = Li ? P.grad[1] : P.grad[0];
  const float lci = Li ? P.lapc[1] : P.lapc[0];
  const float iV = fri.x, pdi = fri.y;
  float tsum = 0.0f, csum = 0.0f;  // component l: finished cells, the current cell
  int last_o = -1;                 // cell of the pair before this round's first

  // one round: this lane's pair `ent` (if has), the particle's np pairs in lanes 0 .. np-1
  auto round = [&](uint ent, bool has, uint np) {
    float ax = 0.0f, ay = 0.0f, az = 0.0f, bx = 0.0f, by = 0.0f, bz = 0.0f;
    float sx = 0.0f, sy = 0.0f, sz = 0.0f, sw = 0.0f;
    const int eo = (int)(ent >> 27);
    const uint j = has ? ent & 0x7ffffffu : ic;
    const float4 pj = pos[j];
    const float4 *rec = frec + 3 * (size_t)j;
    const float4 r0 = rec[0];
    float qx = 0.0f, qy = 0.0f, ejz = 0.0f;
    if (D3) {
      const float *rl = reinterpret_cast<const float *>(rec + 1 + Li);
      qx = rl[0];
      qy = rl[1];
      ejz = rl[2];
    }
    const int up = __shfl_up(eo, 1, 64);
    const int prev = l == 0 ? last_o : up;
    const unsigned long long chg = __ballot(has && eo != prev);
    const int lo = __shfl(eo, g0 + (int)(np ? np - 1u : 0u), 64);
    if (np) last_o = lo;
    if (has && (D3 || j != i)) {
      const float rx = pi.x - pj.x, ry = pi.y - pj.y;
      const float rz = D3 ? pi.z - pj.z : 0.0f;
      const float r2 = D3 ? rx * rx + ry * ry + rz * rz : rx * rx + ry * ry;
      const int Lj = lvl_index(pj.w);
      const float rr = sph_sqrt_normal(r2);  // 1e-4 <= r2 < max(h_i^2, h_j^2)
      const float hj = Lj ? P.kernel[1] : P.kernel[0];
      const float mj = Lj ? P.mass[1] : P.mass[0];
      const float k6j = Lj ? P.k6[1] : P.k6[0];
      const float rk6j = Lj ? P.rcp_k6[1] : P.rcp_k6[0];
      const float spj = Lj ? P.spiky[1] : P.spiky[0];
      const float vkj = Lj ? P.visco_k6[1] : P.visco_k6[0];
      const float jV = r0.x;
      const float ikr = hi - rr, jkr = hj - rr;
      float ipk = 0.0f, ivk = 0.0f, jpk = 0.0f, jvk = 0.0f;
      if (ikr > 0) {
        const float a = spi * ikr * ikr;
        ipk = k6_fast ? sph_div_mk(a, k6i, rk6i) : a / k6i;
        ivk = vki * (ikr);
        const float d = k2i - r2;
        if (D3) {
          const float t0 = qx * (d * d);
          sx = t0 * rx;
          sy = t0 * ry;
          sz = t0 * rz;
          sw = qy * d * (r2 - 0.0f * d);
        } else {
          const float t0 = (-1.0f) * gi * jV * (d * d);
          sx = t0 * rx;
          sy = t0 * ry;
          sz = lci * jV * d * (r2 - 0.0f * d);
        }
      }
      if (jkr > 0) {
        const float a = spj * jkr * jkr;
        jpk = k6_fast ? sph_div_mk(a, k6j, rk6j) : a / k6j;
        jvk = vkj * (jkr);
      }
      const float tp = mi * mj * (pdi + r0.y) * (ipk + jpk) / 2;
      ax = -(rx * tp / rr);
      ay = -(ry * tp / rr);
      if (D3) az = -(rz * tp / rr);
      const float tv = (iV * jV) * P.viscosity * (ivk + jvk) / 2;
      bx = (r0.z - evi.x) * tv;
      by = (r0.w - evi.y) * tv;
      if (D3) bz = (ejz - evi.z) * tv;
    } else if (!D3 && has) {  // SPH-2D/sph_system.cu:640 self term
      sz = lci * mi / dp[ic].x * (k2i) * (0.0f - 0.0f * (k2i));
    }
    float2 *const w = reinterpret_cast<float2 *>(&sh[g][0][0]) + l;
    w[0] = make_float2(ax, bx);
    w[GC / 2] = make_float2(ay, by);
    if (D3) w[2 * (GC / 2)] = make_float2(az, bz);
    w[3 * (GC / 2)] = make_float2(sx, 0.0f);
    w[4 * (GC / 2)] = make_float2(sy, 0.0f);
    w[5 * (GC / 2)] = make_float2(sz, 0.0f);
    if (D3) w[6 * (GC / 2)] = make_float2(sw, 0.0f);
    wave_sync();
    const uint flips = l < 3 ? (uint)(chg >> g0) & 0xffu : 0u;
    const float *const v = &sh[g][l < 7 ? l : 0][0];
    float4 x[4];
#pragma unroll
    for (int k = 0; k < 4; k++) x[k] = reinterpret_cast<const float4 *>(v)[k];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const bool f = (flips >> k) & 1u;
      tsum = f ? tsum + csum : tsum;
      csum = f ? 0.0f : csum;
      csum = csum + (k & 1 ? x[k >> 1].z : x[k >> 1].x);
      csum = csum + (k & 1 ? x[k >> 1].w : x[k >> 1].y);
    }
    wave_sync();
  };

  const uint nl = act && nbl ? nbl_cnt[i] : 0u;
  if (nbl && !__any(nl > SPH_NBL_K)) {
    // lanes 0-3 and 4-7 each read one 16-byte group of the list (layout at struct Aux)
    const uint *my = nbl + ((size_t)(l >> 2) * nbl_stride + ic) * 4 + (l & 3);
    const size_t gs = 2 * 4 * (size_t)nbl_stride;
    uint ent = (uint)l < nl ? *my : 0u;
    for (uint k = 0; __any(k < nl); k += GL) {
      const uint cur = ent, nx = k + GL + (uint)l;
      my += gs;
      ent = nx < nl ? *my : 0u;  // the next round's entry, during this round
      round(cur, k + (uint)l < nl, k < nl ? min(nl - k, (uint)GL) : 0u);
    }
  } else {
    // no list (or one that overflowed): the particle's lanes test eight candidates at a time,
    // cell after cell, and queue the pairs in order; a round whenever some queue holds eight
    uint c[3];
    const bool valid = act && cell_of<V>(P, pi.x, pi.y, pi.z, c);
    uint head = 0, cnt = 0;
    auto drain = [&]() {
      const uint np = min(cnt, (uint)GL);
      const bool has = (uint)l < np;
      round(queue[g][(head + (uint)l) % GQ], has, np);
      head = (head + np) % GQ;
      cnt -= np;
    };
    for (int o = 0; o < VT<V>::nnb; o++) {
      uint s = 0, e = 0;
      if (valid) nb_range<V>(P, o, c, cstart, cend, s, e);
      for (; __any(s < e); s += GL) {
        const uint j = s + (uint)l;
        bool hit = false;
        if (s < e && j < e) {
          const float4 pj = pos[j];
          const float rx = pi.x - pj.x, ry = pi.y - pj.y;
          const float rz = D3 ? pi.z - pj.z : 0.0f;
          const float r2 = D3 ? rx * rx + ry * ry + rz * rz : rx * rx + ry * ry;
          const float k2j = lvl_index(pj.w) ? P.k2[1] : P.k2[0];
          const float maxk2 = k2i > k2j ? k2i : k2j;
          hit = (!D3 && j == i) || (r2 < maxk2 && !(r2 < 0.0001f));
        }
        const uint hits = (uint)(__ballot(hit) >> g0) & 0xffu;
        if (hit) queue[g][(head + cnt + (uint)__popc(hits & ((1u << l) - 1u))) % GQ] = pack_entry(o, j);
        cnt += (uint)__popc(hits);
        wave_sync();
        if (__any(cnt >= (uint)GL)) drain();
      }
    }
    while (__any(cnt > 0u)) drain();
  }
  const float sum = l < 3 ? tsum + csum : csum;
  const float sx = __shfl(sum, g0 + 3, 64), sy = __shfl(sum, g0 + 4, 64);
  const float sz = __shfl(sum, g0 + 5, 64), sw = __shfl(sum, g0 + 6, 64);
  if (!act || l >= 4) return;
  float out;
  if (D3) {
    const float nrm = sqrtf(sx * sx + sy * sy + sz * sz);
    float f = 0.0f;
    if (nrm > P.surface_tension) {
      const float cl = P.surf_coef * sw;
      f = cl * (l == 0 ? sx : (l == 1 ? sy : sz)) / nrm;
    }
    out = l == 3 ? nrm : sum + f;
  } else {
    const float nrm = sqrtf(sx * sx + sy * sy);
    float f = 0.0f;
    if (nrm > P.surface_tension) {
      const float cl = P.surf_coef * sz;
      f = cl * (l == 0 ? sx : sy) / nrm;
    }
    out = sum + f;
    if (P.mouse) {  // SPH-2D/sph_system.cu:781-789
      const float xl = pi.x - P.extern_click[0], yl = pi.y - P.extern_click[1];
      if ((xl * xl + yl * yl) <= (P.extern_len * P.extern_len))
        out += (l == 0 ? P.extern_force[0] : P.extern_force[1]) * P.extern_coe;
    }
    if (l == 2) out = 0.0f;
    if (l == 3) out = nrm;
  }
  acc[4 * (size_t)i + l] = out;
}

// ---------------------------------------------------------------------------------------
// Energy: k_energy (sph_kernels.hip) in nine lanes per particle. The pairs are listed in LDS
// in visiting order (EW at a time), evaluated nine at a time, one per lane, and lane c < 4 adds
// component c (the two wavelet sums, by cell; the two velocity transforms) in list order.
// ---------------------------------------------------------------------------------------
constexpr int EW = 128;  // pairs of a particle listed at a time
constexpr int EC = 12;   // words per component: nine values, padded to 16 bytes

template <int V, bool B>
__global__ __launch_bounds__(BLK) void k_energy_fine(
    DevParams P0, const DevParams *__restrict__ Ptab, SceneCnt *scn,
    const uint *__restrict__ slot, const float4 *__restrict__ pos, const float4 *__restrict__ acc,
    float *__restrict__ energy, const uint *__restrict__ cstart, const uint *__restrict__ cend,
    const uint *n_dev, uint n_host, uint *__restrict__ split_bits,
    const float4 *__restrict__ erec) {
  constexpr bool D3 = VT<V>::dim == 3;
  __shared__ __align__(16) uint pre[BLK / 64][FP + 1][28];
  __shared__ uint list[BLK / 64][FP][EW];
  __shared__ __align__(16) float val[BLK / 64][FP + 1][4][EC];
  const uint n = dev_count(n_dev, n_host);
  const uint nvb = (n + FB - 1) / FB;
  if (blockIdx.x >= nvb) return;
  const uint wave = threadIdx.x >> 6;
  const int lane = (int)(threadIdx.x & 63u), q = lane / FL, r = lane % FL;
  const uint i = xcd_block(blockIdx.x, nvb) * FB + wave * FP + (uint)q;
  const bool act = q < FP && i < n;
  const uint ic = act ? i : 0u;
  const __amdgpu_buffer_rsrc_t prs = sph_rsrc(pos, n_host);
  const DevParams &P = scene_params<B>(P0, Ptab, B ? slot[ic] : 0u);
  const float4 pi = pos[ic];
  const int Li = lvl_index(pi.w);
  const int Lk = D3 ? 0 : Li;  // 3D: large kernel for both levels (3D-2 :1199-1209)
  const float ker = Lk ? P.kernel[1] : P.kernel[0];
  const float ker2 = Lk ? P.k2[1] : P.k2[0];
  const float sk = Lk ? P.sqrt_kernel[1] : P.sqrt_kernel[0];
  const float rker = Lk ? P.rcp_kernel[1] : P.rcp_kernel[0];
  const float rsk = Lk ? P.rcp_sqrt_kernel[1] : P.rcp_sqrt_kernel[0];
  const bool div_fast = P.kernel_div_fast != 0;
  const bool unit = ker == 1.0f && sk == 1.0f;
  uint c[3];
  const bool valid = cell_of<V>(P, pi.x, pi.y, pi.z, c);
  const Row R = load_row<V>(P, r, c, act && valid, cstart, cend);
  auto pair = [&](const float4 &pj) {
    const float rx = pi.x - pj.x, ry = pi.y - pj.y;
    const float rz = D3 ? pi.z - pj.z : 0.0f;
    const float r2 = D3 ? rx * rx + ry * ry + rz * rz : rx * rx + ry * ry;
    return r2 < ker2 && !(D3 && r2 < 0.0001f);  // 3D: also leaves out j == i
  };
  const bool wide = __any(R.e - R.s > 64u);
  unsigned long long m = 0ull;
  uint cn[3] = {0u, 0u, 0u}, base[3], tot;
  if (!wide) {
    m = run_mask(prs, R.s, R.e, pair);
    if (!D3 && i >= R.s && i < R.e) m &= ~(1ull << (i - R.s));
    const unsigned long long l1 = low_bits(R.b1 - R.s), l2 = low_bits(R.b2 - R.s);
    cn[0] = (uint)__popcll(m & l1);
    cn[1] = (uint)__popcll(m & l2 & ~l1);
    cn[2] = (uint)__popcll(m & ~l2);
  } else {
    for (uint j = R.s; j < R.e; j++) {
      const bool h = pair(pos[j]) && (D3 || j != i);
      const int k = R.cell(j);
#pragma unroll
      for (int t = 0; t < 3; t++) cn[t] += (h && k == t) ? 1u : 0u;
    }
  }
  cell_prefix<D3>(pre[wave][q], r, R, cn, base, tot);
  if (!act) tot = 0u;
  float tsum = 0.0f, csum = 0.0f;  // component r: finished cells, the current cell
  int last_o = -1;
  uint *const my = list[wave][q < FP ? q : 0];
  for (uint w0 = 0; __any(w0 < tot); w0 += EW) {
    uint at[3] = {base[0] - w0, base[1] - w0, base[2] - w0};  // wraps below the window
    auto put = [&](uint j) {
      const int k = R.cell(j);
#pragma unroll
      for (int x = 0; x < 3; x++)
        if (k == x) {
          if (at[x] < (uint)EW) my[at[x]] = pack_entry(R.o[x], j);
          at[x]++;
        }
    };
    if (!wide) {
      for (unsigned long long b = m; b; b &= b - 1ull) put(R.s + (uint)__builtin_ctzll(b));
    } else {
      for (uint j = R.s; j < R.e; j++)
        if (pair(pos[j]) && (D3 || j != i)) put(j);
    }
    wave_sync();
    const uint nw = tot > w0 ? min(tot - w0, (uint)EW) : 0u;
    for (uint k0 = 0; __any(k0 < nw); k0 += FL) {
      const uint k = k0 + (uint)r;
      const bool has = k < nw;
      const uint ent = has ? my[k] : 0u;
      const int eo = (int)(ent >> 27);
      const float4 ej = erec[has ? ent & 0x7ffffffu : ic];  // pos.xy, vel.xy
      const int up = __shfl_up(eo, 1, 64);
      const int prev = r == 0 ? last_o : up;
      const unsigned long long chg = __ballot(has && eo != prev);
      const uint np = k0 < nw ? min(nw - k0, (uint)FL) : 0u;
      const int lo = __shfl(eo, lane - r + (int)(np ? np - 1u : 0u), 64);
      if (np) last_o = lo;
      float tx = 0.0f, ty = 0.0f, ux = 0.0f, uy = 0.0f;
      if (has) {
        const float dx = pi.x - ej.x, dy = pi.y - ej.y;
        if (unit) {
          tx = sph_wavelet_unit(dx);
          ty = sph_wavelet_unit(dy);
          ux = ej.z * tx;
          uy = ej.w * ty;
        } else {
          auto dv = [&](float a, float b, float y) { return div_fast ? sph_div_rn(a, b, y) : a / b; };
          tx = sph_wavelet_unit(dv(dx, ker, rker));
          ty = sph_wavelet_unit(dv(dy, ker, rker));
          ux = dv(ej.z * tx, sk, rsk);
          uy = dv(ej.w * ty, sk, rsk);
        }
      }
      float *const w = &val[wave][q][0][r];
      w[0] = tx;
      w[EC] = ty;
      w[2 * EC] = ux;
      w[3 * EC] = uy;
      wave_sync();
      const uint flips = r < 2 ? (uint)(chg >> (lane - r)) & 0x1ffu : 0u;
      const float *const v = val[wave][q][r < 4 ? r : 0];
      float x[FL];
#pragma unroll
      for (int t = 0; t < FL; t++) x[t] = v[t];
#pragma unroll
      for (int t = 0; t < FL; t++) {
        const bool f = (flips >> t) & 1u;
        tsum = f ? tsum + csum : tsum;
        csum = f ? 0.0f : csum;
        csum = csum + x[t];
      }
      wave_sync();
    }
  }
  const float sum = r < 2 ? tsum + csum : csum;
  const float u = __shfl_down(sum, 2, 64) / sum;  // lanes 0, 1: transformed velocity x, y
  const float uy = __shfl_down(u, 1, 64);
  if (!act || r != 0) return;
  const float e2 = u * u + uy * uy;
  float E;
  if (V == SPH_V3D4) E = 0.5f * (Li ? P.mass[1] : P.mass[0]) * (e2);
  else E = 0.5f * (e2);
  energy[i] = E;
  if (split_bits)  // decide_adaptive_kernel, as k_decide
    flag_split<B>(E * P.co_energy + acc[i].w * P.co_surface > P.split_criteria && Li == 0, slot[i],
                  split_bits, scn);
}

inline dim3 blocks_of(size_t n, int per) { return dim3((uint)((n + per - 1) / per)); }

}  // namespace

#define SPH_FINE(KERNEL, variant, batched, grid, st, ...)                                      \
  do {                                                                                         \
    if (batched) {                                                                             \
      if ((variant) == SPH_V3D2) KERNEL<SPH_V3D2, true><<<grid, dim3(BLK), 0, st>>>(__VA_ARGS__); \
      else if ((variant) == SPH_V3D4) KERNEL<SPH_V3D4, true><<<grid, dim3(BLK), 0, st>>>(__VA_ARGS__); \
    } else {                                                                                   \
      if ((variant) == SPH_V2D) KERNEL<SPH_V2D, false><<<grid, dim3(BLK), 0, st>>>(__VA_ARGS__); \
      else if ((variant) == SPH_V3D2) KERNEL<SPH_V3D2, false><<<grid, dim3(BLK), 0, st>>>(__VA_ARGS__); \
      else KERNEL<SPH_V3D4, false><<<grid, dim3(BLK), 0, st>>>(__VA_ARGS__);                  \
    }                                                                                          \
  } while (0)

void launch_density_fine(int variant, const DevParams &P, DevState s, Aux a, const uint *cstart,
                         const uint *cend, uint n, hipStream_t st, const BatchView *bv,
                         const uint *n_dev) {
  SPH_FINE(k_density_fine, variant, bv != nullptr, blocks_of(n, FB), st, P, bv ? bv->Ptab : nullptr,
           s.slot, s.pos, s.ev, s.dp, reinterpret_cast<float *>(a.frec), cstart, cend, n_dev, n, a.nbl,
           a.nbl_cnt, a.nbl_stride);
}

void launch_force_fine(int variant, const DevParams &P, DevState s, Aux a, const uint *cstart,
                       const uint *cend, uint n, hipStream_t st, const BatchView *bv,
                       const uint *n_dev, bool use_nbl) {
  SPH_FINE(k_force_fine, variant, bv != nullptr, blocks_of(n, GB), st, P, bv ? bv->Ptab : nullptr,
           s.slot, s.pos, s.ev, s.dp, a.frec, reinterpret_cast<float *>(s.acc), cstart, cend, n_dev, n,
           use_nbl ? a.nbl : nullptr, a.nbl_cnt, a.nbl_stride);
}

void launch_energy_fine(int variant, const DevParams &P, DevState s, const uint *cstart,
                        const uint *cend, uint n, hipStream_t st, const BatchView *bv,
                        uint *split_bits, const float4 *erec, const uint *n_dev) {
  SPH_FINE(k_energy_fine, variant, bv != nullptr, blocks_of(n, FB), st, P, bv ? bv->Ptab : nullptr,
           bv ? bv->scn : nullptr, s.slot, s.pos, s.acc, s.energy, cstart, cend, n_dev, n, split_bits,
           erec);
}
