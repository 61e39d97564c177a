// Many meshes, one traversal launch (gfx950).
//
// The queries of all items (item = one query array against one mesh) form one flat index
// space. The pipeline:
//   1. keys: item id in the high bits, the query's Hilbert index (in a box around the
//      item's mesh) in the low bits; one stable radix sort then orders every item's queries along
//      the curve and keeps the items apart;
//   2. batch32: a packet = up to 64 consecutive (sorted) queries of one item, one per lane of a
//      wavefront; a packet table (built on the host, most expensive meshes first) maps each
//      wavefront to (item, first query). The wavefront loads its item and mesh records with
//      scalar loads and runs the same packet traversal as the single-mesh kernel, so every
//      wavefront works on one mesh while different wavefronts of a launch work on different
//      meshes. In smaller plans long walks are handed on (batch_items, batch_resolve);
//   3. batch64: the near-surface queries were listed in packet order; a wavefront takes up to 64
//      list entries and decides them in FP64, one of their items after the other (band_walk).
#include "kernels.hpp"
#include "sfc_dev.hpp"
#include "traverse_dev.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>

namespace ebgpu {

namespace {

using namespace dev;

// Item of flat query g (items[lo].base <= g < items[lo + 1].base): binary search over the item
// bases; with a wave-uniform g the probes are scalar loads.
__device__ __forceinline__ uint32_t item_of(const BatchItemDev* __restrict__ items, uint32_t num_items, uint64_t g)
{
  uint32_t lo = 0, hi = num_items;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (items[mid].base <= g) lo = mid;
    else hi = mid;
  }
  return lo;
}

// Sort key of flat query g: (item << 24) | 24-bit Hilbert index of the query on a 256^3 grid of
// the item's box (the mesh box grown by 25%; 8 bits per axis order 64-query packets well at any
// item size). The item of the wavefront's first and last query is searched once per
// wavefront; lanes of a wavefront that straddles items step forward from the first.
template <class KeyT>
__global__ __launch_bounds__(256) void batch_keys_kernel(const BatchItemDev* __restrict__ items, uint32_t num_items,
                                                         uint64_t total, KeyT* __restrict__ keys)
{
  const uint64_t g0 = (uint64_t)blockIdx.x * 256u + uni(threadIdx.x & ~63u);
  if (g0 >= total) return; // whole wavefront
  const uint64_t g     = g0 + __lane_id();
  const uint64_t glast = min(g0 + 63u, total - 1);
  const uint32_t lo0   = uni(item_of(items, num_items, g0));
  const uint32_t lo1   = uni(item_of(items, num_items, glast));
  uint32_t       lo    = lo0;
  if (lo1 != lo0)
    while (lo < lo1 && items[lo + 1].base <= g) lo++;
  if (g >= total) return;
  const BatchItemDev& it = items[lo];
  const uint64_t      j  = g - it.base;
  uint32_t            x[3];
#pragma unroll
  for (int c = 0; c < 3; c++)
    x[c] = (uint32_t)fminf(fmaxf((it.pts[3 * j + c] - it.box_lo[c]) * it.box_inv[c], 0.0f), 255.0f); // NaN -> 0
  keys[g] = KeyT(((uint64_t)lo << 24) | hilbert_index<8>(x[0], x[1], x[2]));
}

// A lane's query of packet p (item it, first query `first`): its index in the item and its point in
// the walk's units. False: no query, or a NaN coordinate (no closest triangle; nothing is written).
__device__ __forceinline__ bool batch_query(const BatchArgs& a, const BatchItemDev& it, const MeshDev& m, uint32_t first,
                                            uint32_t& qi, float& px, float& py, float& pz)
{
  const uint32_t j = first + __lane_id();
  qi               = 0;
  px = py = pz = 0.0f;
  if (j >= it.n) return false;
  qi = a.sorted ? (uint32_t)(a.sorted[it.base + j] - it.base) : j;
  px = it.pts[3 * (size_t)qi] * m.scale;
  py = it.pts[3 * (size_t)qi + 1] * m.scale;
  pz = it.pts[3 * (size_t)qi + 2] * m.scale;
  if (px == px && py == py && pz == pz) return true;
  px = py = pz = 0.0f;
  return false;
}

// The end of a packet: classify, sign and write each lane's closest triangle, and the packet's
// recheck mask. Point and distance^2 in the walk's units.
__device__ __forceinline__ void batch_finish(const BatchArgs& a, const BatchItemDev& it, const MeshDev& m, uint32_t p,
                                             bool active, uint32_t qi, float px, float py, float pz, float best,
                                             uint32_t btri)
{
  px *= m.inv_scale;
  py *= m.inv_scale;
  pz *= m.inv_scale;
  best *= m.inv_scale * m.inv_scale;
  const bool found = active && btri != kInvalid;
  float      d     = 0.0f;
  if (found) {
    const uint32_t feat = closest_feature(m, btri, px, py, pz, best);
    d            = resolve32(m, btri, feat, best, px, py, pz);
    it.out[qi]   = d;
    if (it.tri) it.tri[qi] = m.tris[btri].face;
  }
  if (a.recheck_mask) {
    const uint64_t mask = ballot(found && fabsf(d) < it.recheck_abs);
    if (__lane_id() == 0) a.recheck_mask[p] = mask;
  }
}

// One packet: the wavefront's 64 queries of one item against its mesh. HAND: a long walk is handed
// on (HandOn).
template <int NB, bool COUNT, bool HAND>
__device__ __forceinline__ void batch_packet(const BatchArgs& a, uint32_t p, PairLds* pl)
{
  const SWords<4>    pk = sload<4>(a.packets + 4 * (size_t)p);
  const BatchItemDev it = sload_record(a.items + pk.w[0]);
  const MeshDev      m  = sload_record(a.meshes + it.mesh);
  uint32_t           qi;
  float              px, py, pz;
  const bool         active = batch_query(a, it, m, pk.w[1], qi, px, py, pz);
  float              best = INFINITY, bound = active ? INFINITY : -1.0f;
  uint32_t           btri = kInvalid, n_inner = 0, n_tris = 0, w_inner = 0, w_tris = 0;
  PairCounts         pc{0u, 0u, 0u, 0u};
  Walk<NB>           wk;
  wk.start(0u, 0u);
  uint32_t budget = HAND ? a.hand.budget[0] : ~0u;
  for (;;) {
    mesh_walk<NB, COUNT, HAND>(m, wk, budget, HAND ? a.hand.spread[0] : 0, px, py, pz, bound, best, btri, n_inner, n_tris,
                               w_inner, w_tris, pl, &pc);
    if (!HAND || wk.top == 0) break;
    if (hand_on(a.hand, wk, p, best, btri) != kInvalid) return; // whole wavefront
    budget = ~0u;
  }
  batch_finish(a, it, m, p, active, qi, px, py, pz, best, btri);
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

// The items handed on, as sdf32_items_kernel: stage 0 hands on again, stage 1 walks to the end.
template <int NB, int STAGE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NB == 1 ? 8 : (NB == 2 ? 6 : 4)))) void batch_items_kernel(const BatchArgs a)
{
  const uint32_t wave = uni(threadIdx.x >> 6);
  extern __shared__ PairLds pair_lds[];
  PairLds* const pl = &pair_lds[wave];
  const uint32_t n  = min(a.hand.counts[1 + STAGE], a.hand.item_cap);
  for (uint32_t w = uni(blockIdx.x * 4u + wave); w < n; w += gridDim.x * 4u) {
    const SWords<4> hi = sload<4>(a.hand.items[STAGE] + w);
    if (hi.w[0] == kInvalid) continue;
    const uint32_t      slot = hi.w[0];
    const SWords<4>     pk   = sload<4>(a.packets + 4 * (size_t)uni(a.hand.list[slot]));
    const BatchItemDev  it   = sload_record(a.items + pk.w[0]);
    const MeshDev       m    = sload_record(a.meshes + it.mesh);
    unsigned long long* keys = a.hand.keys + 64 * (size_t)slot + __lane_id();
    const uint64_t      key  = *keys;
    uint32_t            qi;
    float               px, py, pz;
    const bool          active = batch_query(a, it, m, pk.w[1], qi, px, py, pz);
    float               best = __uint_as_float((uint32_t)(key >> 32)), bound = active ? best : -1.0f;
    uint32_t            btri = (uint32_t)key, n_inner = 0, n_tris = 0, w_inner = 0, w_tris = 0;
    Walk<NB>            wk;
    wk.start(hi.w[1], hi.w[2]);
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

// The handed-on packets' end, from their keys.
__global__ __launch_bounds__(256) void batch_resolve_kernel(const BatchArgs a)
{
  const uint32_t n = min(a.hand.counts[0], a.hand.slot_cap);
  for (uint32_t s = uni(blockIdx.x * 4u + (threadIdx.x >> 6)); s < n; s += gridDim.x * 4u) {
    const uint32_t p = uni(a.hand.list[s]);
    if (p == kInvalid) continue;
    const SWords<4>    pk = sload<4>(a.packets + 4 * (size_t)p);
    const BatchItemDev it = sload_record(a.items + pk.w[0]);
    const MeshDev      m  = sload_record(a.meshes + it.mesh);
    uint32_t           qi;
    float              px, py, pz;
    const bool         active = batch_query(a, it, m, pk.w[1], qi, px, py, pz);
    const uint64_t     key    = a.hand.keys[64 * (size_t)s + __lane_id()];
    batch_finish(a, it, m, p, active, qi, px, py, pz, __uint_as_float((uint32_t)(key >> 32)), (uint32_t)key);
  }
}

// PERSIST = false: one wavefront per packet (the early list first, then the table without the
// early packets). PERSIST = true: a grid that fits the device at once; each wavefront takes queue
// entries in the same order until the queue is exhausted (no wavefront waits on another).
template <int NB, bool COUNT, bool PERSIST, bool HAND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NB == 1 ? 8 : (NB == 2 ? 6 : 4)))) void batch32_kernel(const BatchArgs a)
{
  extern __shared__ PairLds pair_lds[]; // one per wavefront of the workgroup
  PairLds* const pl = &pair_lds[uni(threadIdx.x >> 6)];
  if constexpr (PERSIST) {
    const uint32_t ne   = a.early_blocks ? min(*a.early_count, a.early_cap) : 0u;
    const uint32_t skip = a.early_blocks ? a.early_cap : 0u; // queue entries before the table
    for (;;) {
      uint32_t w = 0;
      if (__lane_id() == 0) w = atomicAdd(a.queue, 1u);
      w = uni(rdlane(w, 0));
      if (w >= a.queue_total) return; // whole wavefront
      uint32_t p;
      if (w < skip) {
        if (w >= ne) continue;
        p = uni(a.early_list[w]);
      }
      else {
        p = w - skip;
        if (p >= a.num_packets || (a.early_blocks && a.flag[p])) continue;
      }
      batch_packet<NB, COUNT, HAND>(a, p, pl);
    }
  }
  else {
    const uint32_t wpb = blockDim.x >> 6;
    // wave-uniform, and known to be: the packet and mesh records below are then scalar loads.
    // Plain dispatch order (no XCD remap): all XCDs work on the same stretch of the LPT-ordered
    // packet table, so the meshes in flight at any time are few and stay in the Infinity Cache;
    // with a contiguous eighth of the table per XCD, eight stretches of meshes were in flight and
    // the launch took 2.5x as long (163 against 66 ms on the 256-mesh workload).
    uint32_t w = uni(blockIdx.x * wpb + (threadIdx.x >> 6));
    uint32_t p;
    if (a.early_blocks) {
      // the early packets first (they run longest), then the table in order without them
      const uint32_t ew = a.early_blocks * wpb;
      if (w < ew) {
        if (w >= min(*a.early_count, a.early_cap)) return; // whole wavefront
        p = uni(a.early_list[w]);
      }
      else {
        p = w - ew;
        if (p >= a.num_packets || a.flag[p]) return; // whole wavefront
      }
    }
    else p = w;
    if (p >= a.num_packets) return; // whole wavefront (p is wave-uniform)
    batch_packet<NB, COUNT, HAND>(a, p, pl);
  }
}

// One wavefront per `width` consecutive entries of the recheck list (packet << 6 | lane, in packet
// order: neighbouring queries, mostly of one item). The wavefront takes the distinct items of its
// entries in turn; each listed query is decided in FP64 from its FP32 distance (band_walk).
template <int NB>
__device__ __forceinline__ void batch64_group(const BatchArgs& a, uint32_t count, uint32_t g, uint32_t width, BandLds& L)
{
  const uint32_t lane   = __lane_id();
  const uint32_t e      = g * width + lane;
  const bool     listed = lane < width && e < count;
  uint32_t       item = kInvalid, j = 0;
  if (listed) {
    const uint32_t en  = a.recheck_list[e];
    const size_t   pkt = en >> 6;
    item               = a.packets[4 * pkt];
    j                  = a.packets[4 * pkt + 1] + (en & 63u);
  }
  uint64_t pending = ballot(listed);
  while (pending) {
    const uint32_t cur  = rdlane(item, __ffsll((unsigned long long)pending) - 1);
    const bool     mine = listed && item == cur;
    pending &= ~ballot(mine);
    const BatchItemDev it = sload_record(a.items + cur);
    const MeshDev      m  = sload_record(a.meshes + it.mesh);
    uint32_t           qi = 0;
    float              px = 0.0f, py = 0.0f, pz = 0.0f, d32 = 0.0f;
    if (mine) {
      qi  = a.sorted ? (uint32_t)(a.sorted[it.base + j] - it.base) : j;
      px  = it.pts[3 * (size_t)qi];
      py  = it.pts[3 * (size_t)qi + 1];
      pz  = it.pts[3 * (size_t)qi + 2];
      d32 = it.out[qi];
    }
    const int rep = rep_lane(mine ? 0.0f : -1.0f);
    double    d2;
    uint32_t  tri;
    band_walk<NB>(m, px, py, pz, d32, mine, rdlanef(px, rep), rdlanef(py, rep), rdlanef(pz, rep), L, d2, tri);
    if (mine && tri != kInvalid) {
      it.out[qi] = signed_distance64(m, tri, px, py, pz);
      if (it.tri) it.tri[qi] = m.feat[8 * (size_t)tri + 6];
    }
  }
}

// A fixed grid of wavefronts strides over the groups (their number is only known on the device).
template <int NB>
__global__ __launch_bounds__(256) void batch64_kernel(const BatchArgs a)
{
  __shared__ BandLds lds[4];
  const uint32_t count  = *a.recheck_count;
  const uint32_t waves  = gridDim.x * 4u;
  uint32_t       width  = 64u; // entries per wavefront: fewer when the list is short
  while (width > 1u && count <= width / 2u * min(waves, (uint32_t)kNarrowPackets)) width /= 2u;
  const uint32_t groups = (count + width - 1u) / width;
  for (uint32_t g = uni(blockIdx.x * 4u + (threadIdx.x >> 6)); g < groups; g += waves) 
    batch64_group<NB>(a, count, g, width, lds[uni(threadIdx.x >> 6)]);
}

// One wavefront per packet: the largest cost-grid value over its queries' cells in its mesh's
// grid decides whether it is listed as early.
__global__ __launch_bounds__(256) void batch_mark_kernel(const BatchArgs a)
{
  const uint32_t p = uni(blockIdx.x * 4u + (threadIdx.x >> 6));
  if (p >= a.num_packets) return; // whole wavefront
  const SWords<4>    pk   = sload<4>(a.packets + 4 * (size_t)p);
  const uint32_t     item = pk.w[0], first = pk.w[1];
  const BatchItemDev it   = sload_record(a.items + item);
  const GridDev      gd   = sload_record(a.grids + it.mesh);
  const uint32_t     lane = __lane_id();
  const uint32_t     j    = first + lane;
  uint32_t           c    = 0;
  if (gd.threshold != kInvalid && j < it.n) {
    const uint32_t qi = a.sorted ? (uint32_t)(a.sorted[it.base + j] - it.base) : j;
    uint32_t       cell[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const float x = (it.pts[3 * (size_t)qi + k] - gd.lo[k]) * gd.scale[k];
      cell[k]       = (uint32_t)fminf(fmaxf(x, 0.0f), float(gd.g - 1)); // NaN -> 0
    }
    c = gd.cost[((size_t)cell[2] * gd.g + cell[1]) * gd.g + cell[0]];
  }
  const uint32_t est  = wave_max_u32(c);
  uint32_t       slot = kInvalid;
  if (gd.threshold != kInvalid && est >= gd.threshold && lane == 0) slot = atomicAdd(a.early_count, 1u);
  slot             = rdlane(slot, 0);
  const bool early = slot < a.early_cap;
  if (lane == 0) {
    if (early) a.early_list[slot] = p;
    a.flag[p] = early ? 1 : 0;
  }
}

// launch shape: PERSIST and HAND are the plan's, counting launches hand nothing on
template <int NB, bool PERSIST>
auto batch32_of(bool count, bool hand)
{
  return count ? batch32_kernel<NB, true, PERSIST, false>
               : (hand ? batch32_kernel<NB, false, PERSIST, true> : batch32_kernel<NB, false, PERSIST, false>);
}

template <int NB>
hipError_t launch32(const BatchArgs& a, int wg, bool count, hipStream_t s)
{
  const size_t   lds  = (size_t)(wg / 64) * sizeof(PairLds);
  const uint32_t wpb  = (uint32_t)wg / 64u;
  const bool     hand = a.hand.slot_cap != 0 && !count;
  if (hand && (!a.hand.list || !a.hand.keys || !a.hand.items[0] || !a.hand.items[1] || !a.hand.counts))
    return hipErrorInvalidValue;
  if (a.persist_blocks) {
    if (!a.queue) return hipErrorInvalidValue;
    hipLaunchKernelGGL((batch32_of<NB, true>(count, hand)), dim3(a.persist_blocks), dim3(wg), lds, s, a);
  }
  else {
    const uint32_t blocks = (a.num_packets + wpb - 1) / wpb + a.early_blocks;
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL((batch32_of<NB, false>(count, hand)), dim3(blocks), dim3(wg), lds, s, a);
  }
  if (hand) {
    const size_t   l4 = 4 * sizeof(PairLds);
    const uint32_t g  = std::clamp<uint32_t>(2u * a.num_packets, 512u, 2048u);
    hipLaunchKernelGGL((batch_items_kernel<NB, 0>), dim3(g), dim3(256), l4, s, a);
    hipLaunchKernelGGL((batch_items_kernel<NB, 1>), dim3(g), dim3(256), l4, s, a);
    hipLaunchKernelGGL(batch_resolve_kernel, dim3(std::min(g, (a.hand.slot_cap + 3u) / 4u)), dim3(256), 0, s, a);
  }
  return hipGetLastError();
}

template <int NB>
hipError_t persist_blocks(int wg, bool count, bool hand, uint32_t* blocks)
{
  int          nb = 0, dev = 0, cus = 0;
  const size_t lds = (size_t)(wg / 64) * sizeof(PairLds);
  hipError_t   e   = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, batch32_of<NB, true>(count, hand), wg, lds);
  if (e != hipSuccess) return e;
  if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
  if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
  *blocks = (uint32_t)(std::max(nb, 1) * std::max(cus, 1));
  return hipSuccess;
}

template <int NB>
hipError_t launch64(const BatchArgs& a, hipStream_t s)
{
  if (a.num_packets == 0 || !a.recheck_list) return hipSuccess;
  hipLaunchKernelGGL((batch64_kernel<NB>), dim3(std::min<uint32_t>(16u * a.num_packets, 2048u)), dim3(256), 0, s,
                     a);
  return hipGetLastError();
}

} // namespace

hipError_t launch_batch_keys(const BatchItemDev* items, uint32_t num_items, uint64_t total, void* keys, bool narrow,
                             hipStream_t s)
{
  if (total == 0) return hipSuccess;
  if (narrow && num_items > 256) return hipErrorInvalidValue;
  const dim3 grid((uint32_t)((total + 255) / 256));
  if (narrow)
    hipLaunchKernelGGL((batch_keys_kernel<uint32_t>), grid, dim3(256), 0, s, items, num_items, total,
                       static_cast<uint32_t*>(keys));
  else
    hipLaunchKernelGGL((batch_keys_kernel<uint64_t>), grid, dim3(256), 0, s, items, num_items, total,
                       static_cast<uint64_t*>(keys));
  return hipGetLastError();
}

hipError_t launch_batch_mark(const BatchArgs& a, hipStream_t s)
{
  if (a.num_packets == 0) return hipSuccess;
  if (!a.grids || !a.flag || !a.early_list || !a.early_count) return hipErrorInvalidValue;
  hipLaunchKernelGGL(batch_mark_kernel, dim3((a.num_packets + 3) / 4), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_batch32(const BatchArgs& a, int banks, int wg, bool count, hipStream_t s)
{
  if (wg != 64 && wg != 128 && wg != 256) return hipErrorInvalidValue;
  if (a.early_blocks && (!a.flag || !a.early_list || !a.early_count)) return hipErrorInvalidValue;
  if (banks <= 1) return launch32<1>(a, wg, count, s);
  if (banks == 2) return launch32<2>(a, wg, count, s);
  return launch32<4>(a, wg, count, s);
}

hipError_t batch32_persistent_blocks(int banks, int wg, bool count, bool hand, uint32_t* blocks)
{
  if (wg != 64 && wg != 128 && wg != 256) return hipErrorInvalidValue;
  if (banks <= 1) return persist_blocks<1>(wg, count, hand, blocks);
  if (banks == 2) return persist_blocks<2>(wg, count, hand, blocks);
  return persist_blocks<4>(wg, count, hand, blocks);
}

hipError_t launch_batch64(const BatchArgs& a, int banks, hipStream_t s)
{
  if (banks <= 1) return launch64<1>(a, s);
  if (banks == 2) return launch64<2>(a, s);
  return launch64<4>(a, s);
}

} // namespace ebgpu
