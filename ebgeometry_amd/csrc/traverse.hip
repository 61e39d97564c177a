// Packet (wavefront-coherent) BVH traversal for batched signed-distance queries, gfx950.
//
// One query per lane; the 64 lanes of a wavefront walk the tree together:
//   * the traversal stack is wave-uniform and lives in VGPR lanes (entry j of the stack is
//     lane j%64 of bank j/64), pushed with v_writelane and popped with v_readlane, so it costs
//     no LDS and no scratch;
//   * a node or triangle record is fetched once per wavefront with scalar loads into SGPRs
//     and every lane tests its own query against it;
//   * a child is pushed when its bound (a cylinder along the patch of surface it holds, or a box:
//     WalkNode) is within any lane's cull radius (ballot); children are ordered by the distance
//     seen by the packet's middle lane (to the box, or to the cylinder's centre; nearest popped
//     first), which is the reference's descending-d^2 push order
//     (Source/EBGeometry_BVHImplem.hpp:1178-1194) applied to the packet;
//   * on pop, each lane re-tests the entry's bound against its current cull radius (the
//     reference's `entry.dist2 > curBest2` check, :1145-1149); the entry is skipped when no lane
//     needs it.
// The cylinders took the 16M-query launch on the 327,680-face displaced sphere (K = 4, leaves of 16)
// from 11.0 to 4.86 ms a pass, 1M queries on the 20,480-face unit sphere from 4.98 to 1.01 ms and 1M
// closest faces on an 81,920-face sphere from 10.8 to 2.8 ms.
// Queries arrive presorted along a Hilbert curve, so the 64 queries of a wave are spatial
// neighbours and visit nearly the same nodes.
//
// The per-triangle math follows TriangleSoAT::signedDistanceLane
// (Source/EBGeometry_TriangleSoAImplem.hpp:1199-1293): face region when the three signs of
// (e_i x n).(p - v_i) agree, else the closest of the three vertices and of the edges with
// t in (0,1); the sign comes from the pseudo-normal of the chosen feature. The FP32 pass tracks
// squared distance and the feature; the sign is resolved once per query at the end. The FP64
// pass decides near-surface queries, and closest faces, in double with the reference's formulas (band_walk).
#include "kernels.hpp"
#include "traverse_dev.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>

namespace ebgpu {

namespace {

using namespace dev;

// Workgroups of a list-driven launch (8 per CU); each strides over the list.
constexpr uint32_t kListGrid = 2048;

// Launch modes of the FP32 pass (distinct kernels, so that profiles separate them):
//   kPlain     every query, unseeded
//   kSeeded    every query, cull radius seed_r[q] (learned or caller-supplied bound), with the
//              unseeded redo of the queries whose radius held no triangle
enum Mode : int
{
  kPlain  = 0,
  kSeeded = 1
};

// One packet: the 64 queries pk*64 .. pk*64+63 of the (presorted) query order, one per lane.
template <int NB, bool COUNT, int MODE, bool HAND>
__device__ __forceinline__ void sdf32_packet(const MeshDev& m, const QueryArgs& a, uint64_t n, uint64_t pk, PairLds* pl)
{
  const uint32_t width  = 64u >> a.narrow;
  const uint64_t tid    = pk * width + (uint64_t)__lane_id();
  bool           active = __lane_id() < (int)width && tid < n;
  uint32_t       qi     = 0;
  float          px = 0.0f, py = 0.0f, pz = 0.0f, bound = -1.0f;
  const float    sc = m.scale;
  if (active) {
    qi = a.idx ? a.idx[tid] : (uint32_t)tid;
    px = a.pts[3 * (size_t)qi] * sc;
    py = a.pts[3 * (size_t)qi + 1] * sc;
    pz = a.pts[3 * (size_t)qi + 2] * sc;
    if (MODE == kSeeded) {
      const float r = a.seed_r[qi];
      bound         = r * r * (sc * sc);
    }
    else {
      bound = INFINITY;
    }
    // a NaN coordinate has no closest triangle: its lane takes no part (and writes nothing)
    if (!(px == px && py == py && pz == pz)) {
      px = py = pz = 0.0f;
      bound        = -1.0f;
      active       = false;
    }
  }
  float    best = INFINITY;
  uint32_t btri = kInvalid, n_inner = 0, n_tris = 0, w_inner = 0, w_tris = 0;
  const float seed2 = bound;
  PairCounts pc{0u, 0u, 0u, 0u};
  Walk<NB>   wk;
  wk.start(0u, 0u);
  // A seeded walk is exact only for the lanes that found a triangle within their seed: for the
  // others, nodes between the seed and the true distance were pruned. Those lanes walk again
  // unseeded (from the distances they have), in the same wavefront, while the others sit it out
  // with bound -1; a rare expensive query is so hidden among the other wavefronts of the launch.
  bool     seeded = MODE == kSeeded, redo = false;
  uint32_t budget = HAND ? a.hand.budget[0] : ~0u;
  [[maybe_unused]] uint32_t s_inner = 0, s_tris = 0; // the seeded walk's counts
  for (;;) {
    mesh_walk<NB, COUNT, HAND>(m, wk, budget, HAND ? a.hand.spread[0] : 0, px, py, pz, bound, best, btri, n_inner, n_tris,
                               w_inner, w_tris, pl, &pc);
    const bool missed = MODE == kSeeded && seeded && active && !(btri != kInvalid && best <= seed2);
    if (HAND && wk.top > 0) {
      const uint64_t mmask = ballot(missed);
      if (mmask) {
        // the pruned part is not on the stack: start over without the seeds
        seeded = false;
        wk.start(0u, 0u);
        if (__lane_id() == 0) atomicAdd(a.fallback_count, (uint32_t)__popcll(mmask));
      }
      if (hand_on(a.hand, wk, (uint32_t)pk, best, btri) != kInvalid) return; // whole wavefront
      if (MODE == kSeeded && !redo && active) bound = best;
      budget = ~0u;
      continue;
    }
    if (MODE != kSeeded) break;
    const uint64_t rmask = ballot(missed);
    if (!rmask) break;
    seeded = false;
    redo   = missed;
    if (__lane_id() == 0) atomicAdd(a.fallback_count, (uint32_t)__popcll(rmask));
    s_inner = n_inner;
    s_tris  = n_tris;
    bound   = redo ? best : -1.0f;
    wk.start(0u, 0u);
  }
  const bool found = active && btri != kInvalid;
  if constexpr (MODE == kSeeded && COUNT) {
    if (ballot(redo) && a.work) { // the redone lanes' counts of their second walk
      const uint64_t fi = wave_sum_u64(redo ? (uint64_t)(n_inner - s_inner) : 0ull);
      const uint64_t ft = wave_sum_u64(redo ? (uint64_t)(n_tris - s_tris) : 0ull);
      if (__lane_id() == 0) {
        atomicAdd(a.work + 6, (unsigned long long)fi);
        atomicAdd(a.work + 7, (unsigned long long)ft);
      }
      if (redo) {
        n_inner = s_inner;
        n_tris  = s_tris;
      }
    }
  }
  // back to the mesh's own units (a power of two: exact)
  px *= m.inv_scale;
  py *= m.inv_scale;
  pz *= m.inv_scale;
  best *= m.inv_scale * m.inv_scale;
  float d = 0.0f;
  if (found) {
    const uint32_t feat = closest_feature(m, btri, px, py, pz, best);
    d                   = resolve32(m, btri, feat, best, px, py, pz);
    a.out_d[qi] = d;
    if (a.out_tri) a.out_tri[qi] = m.tris[btri].face;
  }
  const bool rchk = found && fabsf(d) < a.recheck_abs;
  if (a.recheck_mask) {
    const uint64_t rm = ballot(rchk);
    if (__lane_id() == 0) a.recheck_mask[pk] = rm;
  }
  else if (a.recheck_list) wave_append(rchk, qi, a.recheck_list, a.recheck_count);
  if (COUNT && a.packet_cost && __lane_id() == 0) a.packet_cost[pk] = w_inner + w_tris;
  if (COUNT && a.work) {
    const uint64_t si = wave_sum_u64(active ? (uint64_t)n_inner : 0ull);
    const uint64_t st = wave_sum_u64(active ? (uint64_t)n_tris : 0ull);
    if (__lane_id() == 0) {
      atomicAdd(a.work, (unsigned long long)si);
      atomicAdd(a.work + 1, (unsigned long long)st);
      atomicAdd(a.work + 4, (unsigned long long)w_inner);
      atomicAdd(a.work + 5, (unsigned long long)w_tris);
      if (a.pair_work) {
        atomicAdd(a.pair_work, (unsigned long long)pc.pairs);
        atomicAdd(a.pair_work + 1, (unsigned long long)pc.batches);
        atomicAdd(a.pair_work + 2, (unsigned long long)pc.groups);
        atomicAdd(a.pair_work + 3, (unsigned long long)pc.leaves);
      }
    }
  }
}

// One split item: subtree root r for the 64 queries of listed packet j, unseeded; each lane's
// (d^2, triangle) is folded into the packet's keys. d^2 >= 0, so its bits order like the value;
// on equal d^2 the lower triangle index wins.
template <int NB, bool COUNT>
__device__ __forceinline__ void split_item(const MeshDev& m, const QueryArgs& a, uint32_t j, uint32_t r, PairLds* pl)
{
  const uint64_t pk     = a.split_list[j];
  const uint32_t lane   = __lane_id();
  const uint64_t tid    = pk * 64u + lane;
  bool           active = tid < a.n;
  float          px = 0.0f, py = 0.0f, pz = 0.0f;
  if (active) {
    const uint32_t qi = a.idx ? a.idx[tid] : (uint32_t)tid;
    px                = a.pts[3 * (size_t)qi] * m.scale;
    py                = a.pts[3 * (size_t)qi + 1] * m.scale;
    pz                = a.pts[3 * (size_t)qi + 2] * m.scale;
    if (!(px == px && py == py && pz == pz)) { // as in sdf32_packet
      px = py = pz = 0.0f;
      active       = false;
    }
  }
  const SplitRoot rt = sload_record(a.split_roots + r);
  float           best = INFINITY;
  uint32_t        btri = kInvalid, n_inner = 0, n_tris = 0, w_inner = 0, w_tris = 0;
  float           bound = active ? INFINITY : -1.0f;
  Walk<NB>        wk;
  wk.start(rt.ref, rt.cnt);
  mesh_walk<NB, COUNT, false>(m, wk, ~0u, 0, px, py, pz, bound, best, btri, n_inner, n_tris, w_inner, w_tris, pl, nullptr);
  if (active && btri != kInvalid)
    atomicMin(a.split_keys + 64 * (size_t)j + lane, ((unsigned long long)__float_as_uint(best) << 32) | btri);
  if (COUNT && a.work) {
    const uint64_t si = wave_sum_u64(active ? (uint64_t)n_inner : 0ull);
    const uint64_t st = wave_sum_u64(active ? (uint64_t)n_tris : 0ull);
    if (lane == 0) {
      atomicAdd(a.work, (unsigned long long)si);
      atomicAdd(a.work + 1, (unsigned long long)st);
      atomicAdd(a.work + 4, (unsigned long long)w_inner);
      atomicAdd(a.work + 5, (unsigned long long)w_tris);
    }
  }
}

// Grid launch: one wavefront per 64-query packet, 4 packets per workgroup; workgroups are
// mapped XCD-aware so that each XCD works through one contiguous (Morton) range of queries.
// The leading split_blocks workgroups (dispatched first) work through the split items instead,
// beside the packets of the bulk; packets flagged in heavy_flag are skipped.
template <int NB, bool COUNT, int MODE, bool HAND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NB == 1 ? 8 : (NB == 2 ? 6 : 4)))) void sdf32_kernel(const MeshDev m, const QueryArgs a)
{
  const uint32_t wave = uni(threadIdx.x >> 6); // known uniform: list entries load as scalars
  extern __shared__ PairLds pair_lds[];        // one per wavefront
  PairLds* const pl = &pair_lds[wave];
  uint32_t       b = blockIdx.x, nb = gridDim.x;
  if (a.split_blocks) {
    if (b < a.split_blocks) {
      const uint32_t items = min(*a.split_count, a.split_cap) * a.split_nroots;
      for (uint32_t w = b * 4u + wave; w < items; w += a.split_blocks * 4u) {
        const uint32_t j = w / a.split_nroots;
        split_item<NB, COUNT>(m, a, j, w - j * a.split_nroots, pl);
      }
      return;
    }
    b -= a.split_blocks;
    nb -= a.split_blocks;
  }
  if (a.early_blocks) {
    if (b < a.early_blocks) {
      const uint32_t j = b * 4u + wave;
      if (j < min(*a.early_count, a.early_cap)) sdf32_packet<NB, COUNT, MODE, HAND>(m, a, a.n, a.early_list[j], pl);
      return;
    }
    b -= a.early_blocks;
    nb -= a.early_blocks;
  }
  const uint32_t blk = xcd_remap(b, nb);
  const uint64_t n   = a.n;
  const uint64_t pk  = (uint64_t)blk * 4u + wave;
  if (pk * (64u >> a.narrow) >= n) return;      // whole wavefront past the end
  if (a.heavy_flag && a.heavy_flag[pk]) return; // whole wavefront: a split or early packet
  sdf32_packet<NB, COUNT, MODE, HAND>(m, a, n, pk, pl);
}

// The items handed on (HandOn): wavefronts stride over items[STAGE]. Each walks its subtree for the
// 64 queries of the slot's packet from the distances found so far and folds what it finds into
// the keys. d^2 >= 0, so its bits order like the value; on equal d^2 the lower triangle index
// wins, as within a walk. Stage 0 hands on again after budget[1] visits, stage 1 walks to the end.
template <int NB, int STAGE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NB == 1 ? 8 : (NB == 2 ? 6 : 4)))) void sdf32_items_kernel(const MeshDev m, const QueryArgs a)
{
  const uint32_t wave = uni(threadIdx.x >> 6), lane = __lane_id();
  extern __shared__ PairLds pair_lds[];
  PairLds* const pl = &pair_lds[wave];
  const uint32_t n  = min(a.hand.counts[1 + STAGE], a.hand.item_cap);
  for (uint32_t w = uni(blockIdx.x * 4u + wave); w < n; w += gridDim.x * 4u) {
    const SWords<4> it = sload<4>(a.hand.items[STAGE] + w);
    if (it.w[0] == kInvalid) continue;
    const uint32_t      slot = it.w[0];
    const uint32_t      width = 64u >> a.narrow;
    const uint64_t      tid   = (uint64_t)uni(a.hand.list[slot]) * width + lane;
    unsigned long long* keys = a.hand.keys + 64 * (size_t)slot + lane;
    const uint64_t      key  = *keys;
    float               px = 0.0f, py = 0.0f, pz = 0.0f, bound = -1.0f;
    if (lane < width && tid < a.n) {
      const uint32_t qi = a.idx ? a.idx[tid] : (uint32_t)tid;
      px                = a.pts[3 * (size_t)qi] * m.scale;
      py                = a.pts[3 * (size_t)qi + 1] * m.scale;
      pz                = a.pts[3 * (size_t)qi + 2] * m.scale;
      bound             = __uint_as_float((uint32_t)(key >> 32));
      if (!(px == px && py == py && pz == pz)) { // as in sdf32_packet
        px = py = pz = 0.0f;
        bound        = -1.0f;
      }
    }
    float    best = __uint_as_float((uint32_t)(key >> 32));
    uint32_t btri = (uint32_t)key, n_inner = 0, n_tris = 0, w_inner = 0, w_tris = 0;
    Walk<NB> wk;
    wk.start(it.w[1], it.w[2]);
    uint32_t budget = STAGE == 0 ? a.hand.budget[1] : ~0u;
    for (;;) {
      mesh_walk<NB, false, true>(m, wk, budget, a.hand.spread[1], px, py, pz, bound, best, btri, n_inner, n_tris, w_inner,
                                 w_tris, pl, nullptr);
      if (wk.top == 0 || append_items(wk, slot, a.hand.items[1], a.hand.counts + 2, a.hand.item_cap)) break;
      budget = ~0u; // no room: walk on
    }
    const uint64_t now = ((uint64_t)__float_as_uint(best) << 32) | btri;
    if (now < key) atomicMin(keys, (unsigned long long)now);
  }
}

// Wavefronts stride over the listed packets (split or handed on): the winning triangle of each
// query from the packet's keys, as the plain pass ends.
__global__ __launch_bounds__(256) void sdf32_resolve_kernel(const MeshDev m, const QueryArgs a, const uint32_t* list,
                                                            const unsigned long long* result_keys, const uint32_t* count,
                                                            uint32_t cap)
{
  const uint32_t n = min(*count, cap);
  for (uint32_t j = uni(blockIdx.x * 4u + (threadIdx.x >> 6)); j < n; j += gridDim.x * 4u) {
    const uint32_t pk = uni(list[j]);
    if (pk == kInvalid) continue;
    const uint32_t width = 64u >> a.narrow;
    const uint64_t tid   = (uint64_t)pk * width + __lane_id();
    bool           found = false;
    uint32_t       qi    = 0;
    float          d     = 0.0f;
    if (__lane_id() < (int)width && tid < a.n) {
      qi                           = a.idx ? a.idx[tid] : (uint32_t)tid;
      const unsigned long long key = result_keys[64 * (size_t)j + __lane_id()];
      const uint32_t           t   = (uint32_t)key;
      if (t != kInvalid) {
        const float px = a.pts[3 * (size_t)qi], py = a.pts[3 * (size_t)qi + 1], pz = a.pts[3 * (size_t)qi + 2];
        float          d2   = __uint_as_float((uint32_t)(key >> 32)) * (m.inv_scale * m.inv_scale); // the walk's, unscaled
        const uint32_t feat = closest_feature(m, t, px, py, pz, d2);
        d              = resolve32(m, t, feat, d2, px, py, pz);
        a.out_d[qi]    = d;
        if (a.out_tri) a.out_tri[qi] = m.tris[t].face;
        found = true;
      }
    }
    if (a.recheck_mask) {
      const uint64_t rm = ballot(found && fabsf(d) < a.recheck_abs);
      if (__lane_id() == 0) a.recheck_mask[pk] = rm;
    }
    else if (a.recheck_list) wave_append(found && fabsf(d) < a.recheck_abs, qi, a.recheck_list, a.recheck_count);
  }
}

// one wavefront per 64 consecutive packets
__global__ __launch_bounds__(256) void recheck_compact_kernel(const uint64_t* __restrict__ mask, uint64_t npk,
                                                              const uint32_t* __restrict__ idx, uint32_t* __restrict__ list,
                                                              uint32_t* __restrict__ count, uint32_t width)
{
  const uint64_t chunk = (uint64_t)uni(blockIdx.x * 4u + (threadIdx.x >> 6));
  const int      lane  = __lane_id();
  const uint64_t pk    = chunk * 64u + (uint64_t)lane;
  uint64_t       mk    = pk < npk ? mask[pk] : 0ull;
  const uint32_t c     = (uint32_t)__popcll(mk);
  uint32_t       inc   = c;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  const uint32_t total = rdlane(inc, 63);
  if (total == 0) return; // whole wavefront
  uint32_t base = 0;
  if (lane == 0) base = atomicAdd(count, total);
  uint32_t pos = rdlane(base, 0) + inc - c;
  while (mk) {
    const uint64_t tid = pk * width + (uint64_t)(__ffsll((unsigned long long)mk) - 1);
    mk &= mk - 1ull;
    list[pos++] = idx ? idx[tid] : (uint32_t)tid;
  }
}

// The FP64 decision of the closest triangle (band_walk) of one lane's query tid, at most one per
// lane. For ties: the representative point of the 64-query packet (of the presort order, whatever
// the width of the wavefront's) that holds the wavefront's first query: its middle query, or its
// first.
template <int NB>
__device__ __forceinline__ void band_block(const MeshDev& m, const QueryArgs& a, bool active, uint64_t tid0, uint64_t n,
                                           BandLds& L)
{
  const uint64_t tid = tid0 + __lane_id();
  uint32_t       qi  = 0;
  float          px = 0.0f, py = 0.0f, pz = 0.0f, d32 = 0.0f;
  if (active) {
    qi  = a.idx ? a.idx[tid] : (uint32_t)tid;
    px  = a.pts[3 * (size_t)qi];
    py  = a.pts[3 * (size_t)qi + 1];
    pz  = a.pts[3 * (size_t)qi + 2];
    if (!(px == px && py == py && pz == pz)) { // NaN: no closest triangle (sdf32_packet wrote nothing)
      px = py = pz = 0.0f;
      active       = false;
    }
    else d32 = a.out_d[qi];
  }
  const uint64_t g0 = tid0 & ~63ull, rt = g0 + 32u < n ? g0 + 32u : g0;
  const uint32_t rq = a.idx ? a.idx[rt] : (uint32_t)rt;
  double         d2;
  uint32_t       tri;
  band_walk<NB>(m, px, py, pz, d32, active, a.pts[3 * (size_t)rq], a.pts[3 * (size_t)rq + 1], a.pts[3 * (size_t)rq + 2], L,
                d2, tri);
  if (active && tri != kInvalid) {
    a.out_d[qi] = signed_distance64(m, tri, px, py, pz);
    if (a.out_tri) a.out_tri[qi] = m.feat[8 * (size_t)tri + 6];
  }
}

// Every query. The launch lasts as long as the packet with the most triangles in its lanes' bands (next
// to the medial axis), and nothing is handed on here, so packets are narrowed, down to 4 queries, until
// there are kBandPackets of them. Times of the whole call with 64, 32, 16, 8, 4 queries a packet, in us:
// 1M closest faces on 81,920 faces, displaced: 2582, 2198, 2143, 2206, 2748; 100,000 on it: 1953, 1954,
// 1762, 1333, 1186. A mesh without such packets pays for paths that are no longer shared (1M on 4,600
// triangles of a polygon mesh: 1383, 1404, 1558, 1730, 1998; 200,003: 628, 591, 611, 632, 694): the line
// lies where it loses nothing yet.
constexpr uint64_t kBandPackets = 1u << 15;
inline uint32_t    band_narrow(uint64_t n, uint32_t narrow)
{
  while (narrow < 4 && num_packets(n, narrow + 1) <= kBandPackets) narrow++;
  return narrow;
}
template <int NB>
__global__ __launch_bounds__(256) void band_all_kernel(const MeshDev m, const QueryArgs a)
{
  const uint32_t wave = uni(threadIdx.x >> 6), width = 64u >> a.narrow;
  __shared__ BandLds lds[4];
  const uint64_t tid0 = ((uint64_t)xcd_remap(blockIdx.x, gridDim.x) * 4u + wave) * width;
  if (tid0 >= a.n) return; // whole wavefront past the end
  band_block<NB>(m, a, __lane_id() < (int)width && tid0 + __lane_id() < a.n, tid0, a.n, lds[wave]);
}

// A device-side list (a.idx, its length *a.count_ptr): a fixed grid of wavefronts strides over the
// entries, at most 32 per wavefront (the other lanes sit out), fewer when the list is short.
// Near-surface queries are sparse even in presort order, so a wavefront walks several paths, and
// the last to end is the one with the most.
template <int NB>
__global__ __launch_bounds__(256) void band_list_kernel(const MeshDev m, const QueryArgs a)
{
  const uint32_t wave = uni(threadIdx.x >> 6), lane = __lane_id();
  __shared__ BandLds lds[4];
  const uint64_t n     = *a.count_ptr;
  const uint64_t waves = (uint64_t)gridDim.x * 4u;
  uint32_t       width = 32u;
  while (width > 1u && n <= (uint64_t)(width / 2u) * min(waves, (uint64_t)kNarrowPackets)) width /= 2u;
  for (uint64_t w = uni(blockIdx.x * 4u + wave); w * width < n; w += waves)
    band_block<NB>(m, a, lane < width && w * width + lane < n, w * width, n, lds[wave]);
}

template <int NB, int MODE>
void launch32m(const MeshDev& m, const QueryArgs& a, bool count, uint32_t blocks, hipStream_t s)
{
  const size_t lds = 4 * sizeof(PairLds);
  if (count) hipLaunchKernelGGL((sdf32_kernel<NB, true, MODE, false>), dim3(blocks), dim3(256), lds, s, m, a);
  else if (a.hand.slot_cap) hipLaunchKernelGGL((sdf32_kernel<NB, false, MODE, true>), dim3(blocks), dim3(256), lds, s, m, a);
  else hipLaunchKernelGGL((sdf32_kernel<NB, false, MODE, false>), dim3(blocks), dim3(256), lds, s, m, a);
}

template <int NB>
hipError_t launch32(const MeshDev& m, const QueryArgs& a, bool count, hipStream_t s)
{
  const uint32_t blocks = (uint32_t)((num_packets(a.n, a.narrow) + 3) / 4) + a.split_blocks + a.early_blocks;
  if (blocks == 0) return hipSuccess;
  if (a.count_ptr || a.narrow > 6 || (a.narrow && (a.split_blocks || a.early_blocks))) return hipErrorInvalidValue;
  if (a.split_blocks && (!a.split_nroots || !a.split_count || !a.heavy_flag)) return hipErrorInvalidValue;
  if (a.hand.slot_cap && (a.split_blocks || !a.hand.list || !a.hand.keys || !a.hand.items[0] ||
                          !a.hand.items[1] || !a.hand.counts))
    return hipErrorInvalidValue;
  if (a.early_blocks && (!a.early_list || !a.early_count || !a.heavy_flag)) return hipErrorInvalidValue;
  if (a.seed_r) {
    if (!a.fallback_count) return hipErrorInvalidValue;
    launch32m<NB, kSeeded>(m, a, count, blocks, s);
  }
  else {
    launch32m<NB, kPlain>(m, a, count, blocks, s);
  }
  return hipGetLastError();
}

template <int NB>
hipError_t launch64(const MeshDev& m, const QueryArgs& a, hipStream_t s)
{
  if (a.n == 0) return hipSuccess;
  if (a.count_ptr) {
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((a.n + 3) / 4, kListGrid);
    hipLaunchKernelGGL(band_list_kernel<NB>, dim3(blocks), dim3(256), 0, s, m, a);
  }
  else {
    QueryArgs b = a;
    b.narrow    = band_narrow(a.n, a.narrow);
    hipLaunchKernelGGL(band_all_kernel<NB>, dim3((uint32_t)((num_packets(b.n, b.narrow) + 3) / 4)), dim3(256), 0, s, m, b);
  }
  return hipGetLastError();
}

} // namespace

hipError_t launch_sdf32(const MeshDev& m, int banks, const QueryArgs& a, bool count, hipStream_t s)
{
  if (banks <= 1) return launch32<1>(m, a, count, s);
  if (banks == 2) return launch32<2>(m, a, count, s);
  return launch32<4>(m, a, count, s);
}

namespace {

// One wavefront per 64 consecutive packets (packet first + j holds the presorted queries
// (first + j) * 64 ..): packet j is heavy (early) when any of its queries carries the heavy
// (early) cost flag in its sorted presort key; lane j collects packet j's flags, and the
// wavefront appends its heavy and early packets with one atomic per list (one atomic per
// packet on the same two counters cost 0.11 ms at 16M queries).
__global__ __launch_bounds__(256) void heavy_mark_kernel(const HeavyMarkArgs h)
{
  const uint64_t packets = (h.n + 63u) / 64u;
  const uint64_t first   = (uint64_t)uni(blockIdx.x * 4u + (threadIdx.x >> 6)) * 64u;
  if (first >= packets) return; // whole wavefront
  const uint32_t lane = __lane_id();
  const uint64_t lt   = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  uint32_t       mine = 0; // bit 0: heavy flag, bit 1: early flag of packet first + lane
#pragma unroll 8
  for (uint32_t j = 0; j < 64u; j++) {
    const uint64_t tid = (first + j) * 64u + lane;
    const uint32_t key = tid < h.n ? h.skeys[tid] : 0u;
    const bool     hv  = ballot((key >> 31) != 0u) != 0ull;
    const bool     er  = ballot(((key >> 30) & 1u) != 0u) != 0ull;
    if (lane == j) mine = (hv ? 1u : 0u) | (er ? 2u : 0u);
  }
  const uint64_t hmask = ballot((mine & 1u) != 0u);
  uint32_t       hbase = 0;
  if (hmask && lane == 0) hbase = atomicAdd(h.count, (uint32_t)__popcll(hmask));
  const uint32_t hslot = rdlane(hbase, 0) + (uint32_t)__popcll(hmask & lt);
  const bool     heavy = (mine & 1u) && hslot < h.cap;
  const bool     ecand = !heavy && h.early_list && (mine & 2u);
  const uint64_t emask = ballot(ecand);
  uint32_t       ebase = 0;
  if (emask && lane == 0) ebase = atomicAdd(h.early_count, (uint32_t)__popcll(emask));
  const uint32_t eslot = rdlane(ebase, 0) + (uint32_t)__popcll(emask & lt);
  const bool     early = ecand && eslot < h.early_cap;
  const uint64_t pk    = first + lane;
  if (pk < packets) {
    if (heavy) h.list[hslot] = (uint32_t)pk;
    if (early) h.early_list[eslot] = (uint32_t)pk;
    h.flag[pk] = heavy ? 1 : (early ? 2 : 0);
  }
  // reset the 64 result keys of each heavy slot
  for (uint64_t hm = ballot(heavy); hm; hm &= hm - 1ull) {
    const uint32_t sl = rdlane(hslot, __ffsll((unsigned long long)hm) - 1);
    h.keys[64 * (size_t)sl + lane] = ~0ull;
  }
}

} // namespace

hipError_t launch_heavy_mark(const HeavyMarkArgs& h, hipStream_t s)
{
  const uint64_t packets = (h.n + 63) / 64;
  if (packets == 0) return hipSuccess;
  const uint64_t waves = (packets + 63) / 64;
  hipLaunchKernelGGL(heavy_mark_kernel, dim3((uint32_t)((waves + 3) / 4)), dim3(256), 0, s, h);
  return hipGetLastError();
}

hipError_t launch_recheck_compact(const uint64_t* mask, uint64_t n, const uint32_t* idx, uint32_t* list,
                                  uint32_t* count, hipStream_t s, uint32_t narrow)
{
  const uint64_t npk    = num_packets(n, narrow);
  const uint64_t chunks = (npk + 63) / 64;
  if (chunks == 0) return hipSuccess;
  hipLaunchKernelGGL(recheck_compact_kernel, dim3((uint32_t)((chunks + 3) / 4)), dim3(256), 0, s, mask, npk, idx, list,
                     count, 64u >> narrow);
  return hipGetLastError();
}

hipError_t launch_sdf32_resolve(const MeshDev& m, const QueryArgs& a, hipStream_t s)
{
  if (a.split_cap == 0) return hipSuccess;
  hipLaunchKernelGGL(sdf32_resolve_kernel, dim3(std::min((a.split_cap + 3u) / 4u, kListGrid)), dim3(256), 0, s, m, a,
                     a.split_list, a.split_keys, a.split_count, a.split_cap);
  return hipGetLastError();
}

namespace {

// The lists' lengths are only known on the device: fixed grids stride over them.
template <int NB>
hipError_t launch_handed(const MeshDev& m, const QueryArgs& a, hipStream_t s)
{
  const size_t   lds    = 4 * sizeof(PairLds);
  const uint32_t blocks = (uint32_t)std::clamp<uint64_t>((a.n + 255) / 256 * 8u, 512u, kListGrid);
  hipLaunchKernelGGL((sdf32_items_kernel<NB, 0>), dim3(blocks), dim3(256), lds, s, m, a);
  hipLaunchKernelGGL((sdf32_items_kernel<NB, 1>), dim3(blocks), dim3(256), lds, s, m, a);
  hipLaunchKernelGGL(sdf32_resolve_kernel, dim3(std::min(blocks, (a.hand.slot_cap + 3u) / 4u)), dim3(256), 0, s, m, a,
                     a.hand.list, a.hand.keys, a.hand.counts, a.hand.slot_cap);
  return hipGetLastError();
}

} // namespace

hipError_t launch_sdf32_handed(const MeshDev& m, int banks, const QueryArgs& a, hipStream_t s)
{
  if (a.n == 0 || !a.hand.slot_cap) return hipSuccess;
  if (banks <= 1) return launch_handed<1>(m, a, s);
  if (banks == 2) return launch_handed<2>(m, a, s);
  return launch_handed<4>(m, a, s);
}

hipError_t launch_sdf64(const MeshDev& m, int banks, const QueryArgs& a, hipStream_t s)
{
  if (banks <= 1) return launch64<1>(m, a, s);
  if (banks == 2) return launch64<2>(m, a, s);
  return launch64<4>(m, a, s);
}

} // namespace ebgpu
