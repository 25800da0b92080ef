// Split, and the renumbering after merges, over slots (the reference's particle array order).
// The split decisions and the removed entries are bits by slot (a batch: by dense slot, scene
// after scene), so the rank of a slot is a count of the bits before it: a block of 1024 slots
// adds the words before its own itself (up to COUNT_SLOTS slots; at 498k that is 31 kB from L2
// on average), or takes a scan of the blocks' counts. Against a word per slot, a scan of those
// words and a pass over all particles (in cell order, so each reads its slot's word at random):
// split and compaction take 2 launches instead of 7, and a step in which nothing splits or
// merges reads n / 8 bytes for each. 14k particles 118 -> 98 us per step, 498k 749 -> 732. Bound:
// launches; the particle copies when many split.
#include "sph_device.h"

namespace {

// One slot per thread: with four slots to each of 256 threads the loads of one wait for those of
// the one before (split and renumbering, 498k particles 13.8 and 11.1 us against 12.4 and 8.1;
// 126k in a batch 12.8 and 8.3 against 10.3 and 5.3).
constexpr uint SLOT_TILE = 1024;             // slots, and threads, of a block
constexpr uint TILE_WORDS = SLOT_TILE / 32;  // their bit words
// A block sums at most this many slots' words itself: 128 loads per thread in the last block.
// Beyond, three more launches (the blocks' counts and their scan) cost less.
constexpr uint COUNT_SLOTS = 1u << 20;

__global__ __launch_bounds__(BLK) void k_slot_tiles(const uint *__restrict__ bits, uint ntiles,
                                                    uint *__restrict__ tcount) {
  const uint i = blockIdx.x * BLK + threadIdx.x;
  if (i >= ntiles) return;
  const uint4 *const w = reinterpret_cast<const uint4 *>(bits + (size_t)TILE_WORDS * i);
  uint c = 0;
#pragma unroll
  for (uint k = 0; k < TILE_WORDS / 4; k++) {
    const uint4 v = w[k];
    c += __popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w);
  }
  tcount[i] = c;
}

// The block's tile of bits below slot n: its words, the set bits before each word of it (from
// the start of the tile) and, returned, the set bits before the tile; `own` = its own.
struct SlotTile {
  uint word[TILE_WORDS], pre[TILE_WORDS], own, waves[SLOT_TILE / 64];
};
__device__ inline uint load_tile(SlotTile &T, const uint *__restrict__ bits, const uint *__restrict__ toff,
                                 uint tile, uint n) {
  const uint t = threadIdx.x;
  uint part = 0, carry;
  if (!toff) {
    const uint4 *const w = reinterpret_cast<const uint4 *>(bits);
#pragma unroll 4
    for (uint k = t; k < tile * (TILE_WORDS / 4); k += SLOT_TILE) {
      const uint4 v = w[k];
      part += __popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w);
    }
  }
  if (t < 64u) {
    uint v = 0;
    if (t < TILE_WORDS) {
      const uint at = tile * TILE_WORDS + t;
      const uint left = n > at * 32u ? n - at * 32u : 0u;  // slots of the word below n
      v = bits[at] & (left >= 32u ? 0xffffffffu : (1u << left) - 1u);
      T.word[t] = v;
    }
    const uint c = (uint)__popc(v), inc = wave_incl_scan(c, (int)t);
    if (t < TILE_WORDS) T.pre[t] = inc - c;
    if (t == 63u) T.own = inc;
  }
  block_excl_scan(part, T.waves, carry);  // a barrier at least
  return toff ? toff[tile] : carry;
}

__device__ inline uint tiles_of(uint n) { return n ? (n + SLOT_TILE - 1) / SLOT_TILE : 1u; }

// A12 adaptive_particle_kernel (3D-2 :1576-1615; 3D-4 :1583-1656) / split_particle_kernel
// (2D :1092-1131). The parent of rank r (slot order) writes its children at N + r(n-1) + c; only
// the first floor((cap - N) / (n - 1)) flagged parents split. Of a single scene the last block
// also updates the counters (no thread here reads those it writes). s2p: slot -> entry of the
// n_pre particles. qbits (optional): the parents' merge qualification, now that they are small.
// child (optional): entry child[k] of a split parent k receives its (first) child.
template <int V, bool B>
__global__ __launch_bounds__(SLOT_TILE) void k_split(DevParams P0, const DevParams *__restrict__ Ptab,
                                                     const SceneCnt *__restrict__ scn, DevState S, uint n_host,
                                                     const uint *__restrict__ s2p,
                                                           const uint *__restrict__ bits,
                                                     const uint *__restrict__ toff, Counters *cnt,
                                                     uint *__restrict__ qbits, uint *__restrict__ child) {
  constexpr int NS = VT<V>::nsplit;
  __shared__ SlotTile T;
  const uint n = min(cnt->n_pre, n_host), nt = tiles_of(n), tile = blockIdx.x;  // live before the split
  if (tile >= nt) return;
  const uint carry = load_tile(T, bits, toff, tile, n);
  if (!B && tile == nt - 1u && threadIdx.x == 0) {
    const uint total = carry + T.own, room = (P0.cap - n) / (uint)(NS - 1);
    const uint done = total < room ? total : room;
    cnt->s_req = total;
    cnt->s_done = done;
    cnt->n = n + done * (uint)(NS - 1);
    cnt->m = cnt->n;
  }
  if (T.own == 0u) return;
  const uint x = threadIdx.x, word = T.word[x >> 5], bit = x & 31u;
  if (!((word >> bit) & 1u)) return;
  uint rank = carry + T.pre[x >> 5] + (uint)__popc(word & ((1u << bit) - 1u));
  const uint k = s2p[tile * SLOT_TILE + x];
  // base: physical index of the first child; sbase: its slot word
  uint base, sbase;
  const uint w = B ? S.slot[k] : 0u;
  const DevParams &P = scene_params<B>(P0, Ptab, w);
  if (!B) {
    if (rank >= (P.cap - n) / (uint)(NS - 1)) return;
    base = n + rank * (uint)(NS - 1);
    sbase = base;
  } else {
    // children of a batch go after all live entries, scene by scene in parent rank order;
    // their slots continue the scene's own numbering
    const uint sc = w >> SPH_SCENE_SHIFT;
    const SceneCnt &C = scn[sc];
    rank -= C.r0;
    if (rank >= C.s_done) return;
    base = n + (C.done_base + rank) * (uint)(NS - 1);
    sbase = (sc << SPH_SCENE_SHIFT) | (C.n_pre + rank * (uint)(NS - 1));
  }
  const float hs = P.kernel[1] / 2;
  const float4 p = S.pos[k];
  const float4 v = S.vel[k], e = S.ev[k], a = S.acc[k];
  const float2 dpk = S.dp[k];
  const float en = NS == 2 ? S.energy[k] : S.energy[k] / 4;
  const float lev2 = __uint_as_float(2u);
  // children copy every field of the parent (3D leaves dens/press/surface/tension
  // unwritten in the reference; copies make the downloaded state defined)
  const float4 cp[3] = {make_float4(p.x - hs, p.y, p.z, lev2), make_float4(p.x, p.y, p.z - hs, lev2),
                        make_float4(p.x, p.y, p.z + hs, lev2)};
#pragma unroll
  for (int c = 0; c < NS - 1; c++) {
    const uint q = base + c;
    S.pos[q] = cp[c];
    S.vel[q] = v;
    S.ev[q] = e;
    S.acc[q] = a;
    S.dp[q] = dpk;
    S.energy[q] = en;
    S.slot[q] = sbase + c;
  }
  S.pos[k] = make_float4(p.x + hs, p.y, p.z, lev2);
  if (NS != 2) S.energy[k] = en;
  if (child) child[k] = base;
  if (qbits && (VT<V>::dim == 2 || en * P.co_energy + a.w * P.co_surface < P.merge_criteria))
    atomicOr(&qbits[k >> 5], 1u << (k & 31u));
}

// A14 rearrange (SPH-3D-2/sph_system.cu:1818-1840) as a renumbering: survivors get the rank of
// their slot among survivors; removed entries are dropped by the next sort. Bound = cnt->m, the
// entries before the merge. Of a single scene the last block sets the live count (no thread here
// reads it; a batch's compaction plan has set it). s2p: slot -> entry, of all slots (all_slots) or
// of the n_pre particles before the split, whose children sit at their slot (a batch: after all
// n_pre entries, scene by scene).
template <bool B>
__global__ __launch_bounds__(SLOT_TILE) void k_renumber(DevState S, const SceneCnt *__restrict__ scn, uint ns,
                                                        uint per_split, uint n_host,
                                                        const uint *__restrict__ s2p, bool all_slots,
                                                              const uint *__restrict__ bits,
                                                        const uint *__restrict__ toff, Counters *cnt) {
  __shared__ SlotTile T;
  const uint n = min(cnt->m, n_host), nt = tiles_of(n), tile = blockIdx.x;
  if (tile >= nt) return;
  const uint carry = load_tile(T, bits, toff, tile, n);
  if (!B && tile == nt - 1u && threadIdx.x == 0) cnt->n = n - (carry + T.own);
  if (carry + T.own == 0u) return;  // no slot up to here changes
  const uint n_pre = cnt->n_pre;
  const uint x = threadIdx.x, word = T.word[x >> 5], bit = x & 31u;
  const uint d = tile * SLOT_TILE + x;
  if (d >= n) return;
  const uint before = carry + T.pre[x >> 5] + (uint)__popc(word & ((1u << bit) - 1u));
  uint k, to;
  if (!B) {
    k = all_slots || d < n_pre ? s2p[d] : d;
    to = d - before;
  } else {
    uint lo = 0, hi = ns;  // the last scene whose slots start at or before d
    while (hi - lo > 1u) {
      const uint mid = (lo + hi) / 2u;
      if (scn[mid].first2 <= d) lo = mid;
      else hi = mid;
    }
    const SceneCnt &C = scn[lo];
    const uint l = d - C.first2;
    k = l < C.n_pre ? s2p[C.first + l] : n_pre + C.done_base * per_split + (l - C.n_pre);
    to = (lo << SPH_SCENE_SHIFT) | (l - (before - C.a0));
  }
  S.slot[k] = (word >> bit) & 1u ? SPH_DEAD : to;
}

// offsets of the tiles' bits by a scan, or null where the blocks count for themselves
const uint *tile_offsets(const SlotBits &sb, const uint *bits, uint n, hipStream_t st) {
  if (n <= COUNT_SLOTS) return nullptr;
  const uint nt = (n + SLOT_TILE - 1) / SLOT_TILE;
  k_slot_tiles<<<dim3((nt + BLK - 1) / BLK), dim3(BLK), 0, st>>>(bits, nt, sb.toff);
  sph_exclusive_scan(sb.toff, sb.toff, nullptr, nt, nullptr, sb.scan_tmp, st);
  return sb.toff;
}

inline dim3 tile_grid(uint n) { return dim3(n ? (n + SLOT_TILE - 1) / SLOT_TILE : 1u); }

}  // namespace

size_t sph_bit_words(size_t n) { return (n + SLOT_TILE - 1) / SLOT_TILE * TILE_WORDS; }
size_t sph_bit_tiles(size_t n) { return (n + SLOT_TILE - 1) / SLOT_TILE; }

void launch_split(int variant, const DevParams &P, DevState s, uint n, const SlotBits &sb, const uint *s2p,
                  Counters *cnt, hipStream_t st, bool with_qual, const BatchView *bv, uint *child) {
  const uint *toff = tile_offsets(sb, sb.split, n, st);
#define SPH_SPLIT(V, B)                                                                           \
  k_split<V, B><<<tile_grid(n), dim3(SLOT_TILE), 0, st>>>(                                         \
      P, bv ? bv->Ptab : nullptr, bv ? bv->scn : nullptr, s, n, s2p, sb.split, toff, cnt,          \
      with_qual ? sb.qual : nullptr, child)
  if (bv) {
    if (variant == SPH_V3D2) SPH_SPLIT(SPH_V3D2, true);
    else SPH_SPLIT(SPH_V3D4, true);
  } else {
    if (variant == SPH_V2D) SPH_SPLIT(SPH_V2D, false);
    else if (variant == SPH_V3D2) SPH_SPLIT(SPH_V3D2, false);
    else SPH_SPLIT(SPH_V3D4, false);
  }
#undef SPH_SPLIT
}

void launch_renumber(int variant, DevState s, uint m, const SlotBits &sb, const uint *s2p, bool all_slots,
                     Counters *cnt, hipStream_t st, const BatchView *bv) {
  const uint *toff = tile_offsets(sb, sb.dead, m, st);
  const uint per = variant == SPH_V3D4 ? 3u : 1u;
  if (bv)
    k_renumber<true><<<tile_grid(m), dim3(SLOT_TILE), 0, st>>>(s, bv->scn, bv->n_scenes, per, m, s2p, all_slots,
                                                         sb.dead, toff, cnt);
  else
    k_renumber<false><<<tile_grid(m), dim3(SLOT_TILE), 0, st>>>(s, nullptr, 0u, per, m, s2p, all_slots, sb.dead,
                                                          toff, cnt);
}
