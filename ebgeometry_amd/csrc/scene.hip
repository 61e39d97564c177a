// Batched value() of a CSG union scene on gfx950: spheres, axis-aligned boxes and mesh instances
// under similarity transforms, combined by a union over a 4-wide BVH of their bounding boxes.
//
// Semantics follow BVHUnionIF::value (Source/EBGeometry_CSGImplem.hpp:466-501): the running
// value v starts at +inf, a node is visited when its box distance^2 is within max(0, v)^2, and
// each leaf primitive lowers v to min(v, primitive value). Primitive values:
//   sphere  |p - c| - r                                  (AnalyticDistanceFunctions.hpp:240-247)
//   box     min(0, max_i delta_i) + |max(0, delta)|,
//           delta_i = max(lo_i - p_i, p_i - hi_i)        (AnalyticDistanceFunctions.hpp:377-399)
//   mesh    s * mesh(M (p - t) / s), M = Rx Ry Rz        (TransformImplem.hpp:140-270)
// The packet scheme is the one of the mesh kernel: one query per lane, a wave-uniform stack in
// VGPR lanes, records read with scalar loads. A mesh instance that some lane needs is walked by
// the whole wavefront, unseeded (the sign of its value is only known once its nearest triangle
// is); lanes that do not need it carry a negative bound and take no part. In FP32 that walk goes over
// the mesh's cylinder bounds and triangle discs, and the whole wavefront evaluates each triangle that
// some lane may need (wide_walk): with box bounds and spheres the FP32 pass of 4M points against 4096
// spheres, 1024 boxes and 8 meshes of 20,480 faces took 4.14 ms, so 2.80 ms (and less since long walks
// are handed on), and a walk that starts from the running value for lanes outside the mesh's box
// measured the same. The FP64 pass only asks whether an instance comes within the query's |value|:
// 1.85 -> 0.30 ms.
//
// FP32 pass for all queries; an FP64 pass (same traversal in double, FP64 primitive parameters,
// FP64 triangle math) redoes queries with |v| below the recheck threshold, seeded with the FP32
// value plus slack.
#include "kernels.hpp"
#include "traverse_dev.hpp"

#include <hip/hip_runtime.h>

namespace ebgpu {

namespace {

using namespace dev;

template <class R>
__device__ __forceinline__ R sphere_value(R px, R py, R pz, R cx, R cy, R cz, R r)
{
  const R dx = px - cx, dy = py - cy, dz = pz - cz;
  return sqrt(dx * dx + dy * dy + dz * dz) - r;
}

template <class R>
__device__ __forceinline__ R box_value(R px, R py, R pz, R lx, R ly, R lz, R hx, R hy, R hz)
{
  const R dx = max(lx - px, px - hx), dy = max(ly - py, py - hy), dz = max(lz - pz, pz - hz);
  const R ox = max(R(0), dx), oy = max(R(0), dy), oz = max(R(0), dz);
  return min(R(0), max(dx, max(dy, dz))) + sqrt(ox * ox + oy * oy + oz * oz);
}

struct SceneCounts
{
  uint32_t n_inner = 0, n_prims = 0, n_tris = 0, w_inner = 0, w_prims = 0, w_tris = 0;
};

// The point in a mesh instance's own space, FP32 (pr.A = M / s).
__device__ __forceinline__ void instance_point(const PrimRec& pr, float px, float py, float pz, float& qx, float& qy,
                                               float& qz)
{
  const float ux = px - pr.t[0], uy = py - pr.t[1], uz = pz - pr.t[2];
  qx = pr.A[0] * ux + pr.A[1] * uy + pr.A[2] * uz;
  qy = pr.A[3] * ux + pr.A[4] * uy + pr.A[5] * uz;
  qz = pr.A[6] * ux + pr.A[7] * uy + pr.A[8] * uz;
}

// Where a packet's long instance walks are handed on to.
struct SceneHand
{
  const HandOn* h;
  SceneSlot*    slots;
  uint32_t      packet, head; // head: the packet's last slot (kInvalid: none)
};

// Union value of the scene at (px,py,pz) for this lane. v holds the starting value (+inf, or an
// upper bound on the answer when seeded); bound < 0 marks a lane without a query. HAND: instances
// whose walks were handed on are missing from v, which costs the rest of the walk some culling.
template <int KM, int NB, class R, bool COUNT, bool HAND>
__device__ __forceinline__ void scene_traverse(const SceneDev& sc, R px, R py, R pz, R& v, R bound, SceneCounts& c,
                                               SceneHand* hand)
{
  [[maybe_unused]] const R    seed = v; // FP64: a bound on |value| (+inf: none)
  const Node<4>* __restrict__ nodes = static_cast<const Node<4>*>(sc.nodes);
  LaneStack<NB>               st;
  st.init();
  const int  lane   = __lane_id();
  const bool active = bound >= R(0);
  const int  rep    = 0; // the scene tree orders children by the wave minimum
  int        top    = 0;
  Entry      root{0u, 0u, sc.root_lo[0], sc.root_lo[1], sc.root_lo[2], sc.root_hi[0], sc.root_hi[1], sc.root_hi[2]};
  st.put(top++, root);

  while (top > 0) {
    const Entry e    = st.get(--top);
    const R     d2e  = box_d2<R>(px, py, pz, e.lx, e.ly, e.lz, e.hx, e.hy, e.hz);
    const bool  need = d2e <= bound;
    if (ballot(need) == 0) continue;

    if (e.cnt == 0u) {
      if (COUNT) { c.n_inner += need ? 1u : 0u; c.w_inner++; }
      push_children<4, NB, R, true>(sload_record(nodes + uni(e.ref)), px, py, pz, bound, st, top, rep);
      if (top > 64 * NB) { // beyond the build-time worst case: record it, keep what is held
        if (lane == 0 && sc.status) atomicOr(sc.status, kStatusStackOverflow);
        top = 64 * NB;
      }
      continue;
    }
    const uint32_t first = uni(e.ref), cnt = uni(e.cnt);
    for (uint32_t i = first; i < first + cnt; i++) {
      const PrimRec  pr = sload_record(sc.prims + i);
      const bool     pn = box_d2<R>(px, py, pz, pr.bv[0], pr.bv[1], pr.bv[2], pr.bv[3], pr.bv[4], pr.bv[5]) <= bound;
      if (ballot(pn) == 0) continue;
      if (COUNT) { c.n_prims += pn ? 1u : 0u; c.w_prims++; }
      const uint32_t type = uni(pr.type);
      R              val;
      if (type == kPrimSphere) {
        if constexpr (sizeof(R) == 4) val = sphere_value<R>(px, py, pz, pr.a[0], pr.a[1], pr.a[2], pr.a[3]);
        else {
          const PrimRec64 q = sload_record(sc.prims64 + i);
          val               = sphere_value<R>(px, py, pz, q.a[0], q.a[1], q.a[2], q.a[3]);
        }
      }
      else if (type == kPrimBox) {
        if constexpr (sizeof(R) == 4)
          val = box_value<R>(px, py, pz, pr.a[0], pr.a[1], pr.a[2], pr.a[3], pr.a[4], pr.a[5]);
        else {
          const PrimRec64 q = sload_record(sc.prims64 + i);
          val               = box_value<R>(px, py, pz, q.a[0], q.a[1], q.a[2], q.a[3], q.a[4], q.a[5]);
        }
      }
      else {
        const MeshDev  md = sload_record(sc.meshes + uni(pr.mesh));
        R              qx, qy, qz, s;
        if constexpr (sizeof(R) == 4) {
          instance_point(pr, px, py, pz, qx, qy, qz);
          s = pr.s;
        }
        else {
          const PrimRec64 q  = sload_record(sc.prims64 + i);
          const double    ux = px - q.t[0], uy = py - q.t[1], uz = pz - q.t[2];
          s  = q.s;
          qx = (q.A[0] * ux + q.A[1] * uy + q.A[2] * uz) / s;
          qy = (q.A[3] * ux + q.A[4] * uy + q.A[5] * uz) / s;
          qz = (q.A[6] * ux + q.A[7] * uy + q.A[8] * uz) / s;
        }
        // How near the instance must come to matter. FP32: a lane needs the nearest triangle itself
        // (the mesh may hold it inside at any depth). FP64: the pass only decides queries whose
        // value's magnitude is at most seed, so no primitive's value is below -seed and an instance
        // further off than seed is not the minimum.
        R near = R(INFINITY);
        if constexpr (sizeof(R) == 8) {
          const R lim = seed / s * R(1.0 + 0x1p-18) + R(md.hmax) * R(0x1p-18);
          near        = lim * lim;
        }
        near             = pn ? near : R(-1);
        R        best    = INFINITY;
        uint32_t btri    = kInvalid, bfeat = 0;
        if constexpr (sizeof(R) == 4) {
          Walk<NB> wk;
          wk.start(0u, 0u);
          wide_walk<NB, COUNT, HAND>(md, wk, HAND ? hand->h->budget[0] : 0u, HAND ? hand->h->spread[0] : 0, qx, qy, qz, near,
                                     best, btri, c.n_inner, c.n_tris, c.w_inner, c.w_tris);
          if (HAND && wk.top > 0) {
            const uint32_t j = hand_on(*hand->h, wk, hand->packet, pn ? best : -1.0f, btri);
            if (j != kInvalid) {
              if (lane == 0) hand->slots[j] = SceneSlot{hand->packet, i, hand->head, 0u};
              hand->head = j;
              continue;
            }
            // no room: walk on (a lane's bound is its best so far)
            wide_walk<NB, COUNT, false>(md, wk, 0u, 0, qx, qy, qz, pn ? best : -1.0f, best, btri, c.n_inner, c.n_tris,
                                        c.w_inner, c.w_tris);
          }
        }
        else
          traverse64<KM, NB>(md, qx, qy, qz, near, best, btri, bfeat);
        // Lanes that did not ask for this instance (near = -1) or found nothing that near still saw
        // triangles the wavefront evaluated, so their btri names some triangle but not their nearest.
        val = R(INFINITY);
        if (pn && btri != kInvalid && best <= near) {
          if constexpr (sizeof(R) == 4) val = s * resolve32(md, btri, closest_feature(md, btri, qx, qy, qz), best, qx, qy, qz);
          else val = s * resolve64(md, btri, bfeat, best, qx, qy, qz);
        }
      }
      v = min(v, val);
    }
    if (active) {
      const R b = max(R(0), v);
      bound     = b * b;
    }
  }
}

// FP32 pass, one 64-query packet per wavefront, 4 per workgroup, XCD-aware block order. Bound by the
// latency of its scalar loads: registers are held to what 7 wavefronts per SIMD have.
template <int NB, bool COUNT, bool HAND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NB == 1 ? 7 : 4))) void scene32_kernel(
  const SceneDev sc, const QueryArgs a, SceneSlot* const slots)
{
  const uint32_t blk = xcd_remap(blockIdx.x, gridDim.x);
  const uint64_t n   = a.n;
  if ((uint64_t)blk * 256u >= n) return;
  const uint64_t tid    = (uint64_t)blk * 256u + threadIdx.x;
  const bool     active = tid < n;
  uint32_t       qi     = 0;
  float          px = 0.0f, py = 0.0f, pz = 0.0f;
  if (active) {
    qi = a.idx ? a.idx[tid] : (uint32_t)tid;
    px = a.pts[3 * (size_t)qi];
    py = a.pts[3 * (size_t)qi + 1];
    pz = a.pts[3 * (size_t)qi + 2];
  }
  // Seeded (learned bound or caller radii): the walk starts from v = seed, bound seed^2, and is
  // exact when some primitive comes in below the seed; the other lanes redo the walk unseeded
  // in the same wavefront (the rest sit it out with bound -1).
  const float seed = (active && a.seed_r) ? a.seed_r[qi] : INFINITY;
  float       v    = seed;
  SceneCounts c;
  SceneHand   hand{&a.hand, slots, uni(blk * 4u + (threadIdx.x >> 6)), kInvalid};
  scene_traverse<4, NB, float, COUNT, HAND>(sc, px, py, pz, v, active ? seed * seed : -1.0f, c, &hand);
  if (!HAND && a.seed_r) {
    const bool     redo  = active && !(v < seed);
    const uint64_t rmask = ballot(redo);
    if (rmask) {
      float       v2 = INFINITY;
      SceneCounts c2;
      scene_traverse<4, NB, float, COUNT, false>(sc, px, py, pz, v2, redo ? INFINITY : -1.0f, c2, nullptr);
      if (redo) v = v2;
      if (__lane_id() == 0 && a.fallback_count) atomicAdd(a.fallback_count, (uint32_t)__popcll(rmask));
      if (COUNT) {
        c.n_inner += c2.n_inner, c.n_prims += c2.n_prims, c.n_tris += c2.n_tris;
        c.w_inner += c2.w_inner, c.w_prims += c2.w_prims, c.w_tris += c2.w_tris;
      }
    }
  }
  if (active) a.out_d[qi] = v;
  if (HAND && hand.head != kInvalid) { // the value is settled, and checked, when the slots are done
    if (__lane_id() == 0) slots[hand.head].head = 1u;
    return;
  }
  if (a.recheck_list) wave_append(active && fabsf(v) < a.recheck_abs, qi, a.recheck_list, a.recheck_count);
  if (COUNT && a.work) {
    const uint64_t si = wave_sum_u64(active ? (uint64_t)c.n_inner : 0ull);
    const uint64_t st = wave_sum_u64(active ? (uint64_t)c.n_tris : 0ull);
    const uint64_t sp = wave_sum_u64(active ? (uint64_t)c.n_prims : 0ull);
    if (__lane_id() == 0) {
      atomicAdd(a.work, (unsigned long long)si);
      atomicAdd(a.work + 1, (unsigned long long)st);
      atomicAdd(a.work + 4, (unsigned long long)c.w_inner);
      atomicAdd(a.work + 5, (unsigned long long)c.w_tris);
      atomicAdd(a.work + 6, (unsigned long long)sp);
      atomicAdd(a.work + 7, (unsigned long long)c.w_prims);
    }
  }
}

// The handed-on instance walks, as the mesh kernel's items: stage 0 hands on again, stage 1 walks to
// the end.
template <int NB, int STAGE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NB == 1 ? 7 : 4))) void scene_items_kernel(
  const SceneDev sc, const QueryArgs a, const SceneSlot* const slots)
{
  const uint32_t n = min(a.hand.counts[1 + STAGE], a.hand.item_cap);
  for (uint32_t w = uni(blockIdx.x * 4u + (threadIdx.x >> 6)); w < n; w += gridDim.x * 4u) {
    const SWords<4> hi = sload<4>(a.hand.items[STAGE] + w);
    if (hi.w[0] == kInvalid) continue;
    const uint32_t      slot = hi.w[0];
    const SWords<4>     sl   = sload<4>(slots + slot);
    const PrimRec       pr   = sload_record(sc.prims + sl.w[1]);
    const MeshDev       md   = sload_record(sc.meshes + uni(pr.mesh));
    unsigned long long* keys = a.hand.keys + 64 * (size_t)slot + __lane_id();
    const uint64_t      key  = *keys;
    const uint64_t      tid  = 64u * (uint64_t)sl.w[0] + __lane_id();
    float               qx = 0.0f, qy = 0.0f, qz = 0.0f;
    if (tid < a.n) {
      const size_t qi = a.idx ? a.idx[tid] : (uint32_t)tid;
      instance_point(pr, a.pts[3 * qi], a.pts[3 * qi + 1], a.pts[3 * qi + 2], qx, qy, qz);
    }
    float    best = __uint_as_float((uint32_t)(key >> 32)); // -1: a lane without a query
    uint32_t btri = (uint32_t)key, n_inner = 0, n_tris = 0, w_inner = 0, w_tris = 0;
    Walk<NB> wk;
    wk.start(hi.w[1], hi.w[2]);
    wide_walk<NB, false, STAGE == 0>(md, wk, a.hand.budget[1], a.hand.spread[1], qx, qy, qz, best, best, btri, n_inner,
                                     n_tris, w_inner, w_tris);
    if (STAGE == 0 && wk.top > 0 && !append_items(wk, slot, a.hand.items[1], a.hand.counts + 2, a.hand.item_cap))
      wide_walk<NB, false, false>(md, wk, 0u, 0, qx, qy, qz, best, best, btri, n_inner, n_tris, w_inner, w_tris);
    const uint64_t now = ((uint64_t)__float_as_uint(best) << 32) | btri;
    if (now < key) atomicMin(keys, (unsigned long long)now);
  }
}

// The handed-on packets' end: each lane's value is the least of the packet's own and its slots'.
__global__ __launch_bounds__(256) void scene_resolve_kernel(const SceneDev sc, const QueryArgs a,
                                                            const SceneSlot* const slots)
{
  const uint32_t n = min(a.hand.counts[0], a.hand.slot_cap);
  for (uint32_t s = uni(blockIdx.x * 4u + (threadIdx.x >> 6)); s < n; s += gridDim.x * 4u) {
    const uint32_t p = uni(a.hand.list[s]);
    if (p == kInvalid || uni(slots[s].head) == 0u) continue;
    const uint64_t tid    = 64u * (uint64_t)p + __lane_id();
    const bool     active = tid < a.n;
    uint32_t       qi     = 0;
    float          px = 0.0f, py = 0.0f, pz = 0.0f, v = INFINITY;
    if (active) {
      qi = a.idx ? a.idx[tid] : (uint32_t)tid;
      px = a.pts[3 * (size_t)qi];
      py = a.pts[3 * (size_t)qi + 1];
      pz = a.pts[3 * (size_t)qi + 2];
      v  = a.out_d[qi];
    }
    for (uint32_t k = s; k != kInvalid;) {
      const SWords<4> sl   = sload<4>(slots + k);
      const PrimRec   pr   = sload_record(sc.prims + sl.w[1]);
      const MeshDev   md   = sload_record(sc.meshes + uni(pr.mesh));
      const uint64_t  key  = a.hand.keys[64 * (size_t)k + __lane_id()];
      const float     best = __uint_as_float((uint32_t)(key >> 32));
      const uint32_t  btri = (uint32_t)key;
      float           qx, qy, qz;
      instance_point(pr, px, py, pz, qx, qy, qz);
      if (active && best >= 0.0f && btri != kInvalid)
        v = min(v, pr.s * resolve32(md, btri, closest_feature(md, btri, qx, qy, qz), best, qx, qy, qz));
      k = sl.w[2];
    }
    if (active) a.out_d[qi] = v;
    if (a.recheck_list) wave_append(active && fabsf(v) < a.recheck_abs, qi, a.recheck_list, a.recheck_count);
  }
}

// FP64 pass over the recheck list. The seed |v32| (1 + rel) + abs bounds the exact value from
// above, so every primitive that can attain the minimum is visited; the result replaces the
// FP32 value only if some primitive came in at or below the seed.
template <int KM, int NB>
__device__ __forceinline__ void scene64_block(const SceneDev& sc, const QueryArgs& a, uint64_t n, uint64_t tid)
{
  const bool     active = tid < n;
  uint32_t       qi     = 0;
  double         px = 0.0, py = 0.0, pz = 0.0, seed = -1.0;
  if (active) {
    qi   = a.idx ? a.idx[tid] : (uint32_t)tid;
    px   = a.pts[3 * (size_t)qi];
    py   = a.pts[3 * (size_t)qi + 1];
    pz   = a.pts[3 * (size_t)qi + 2];
    seed = a.slack_abs > 0.0f ? fabs((double)a.out_d[qi]) * (1.0 + (double)a.slack_rel) + (double)a.slack_abs
                              : INFINITY;
  }
  double      v = seed;
  SceneCounts c;
  scene_traverse<KM, NB, double, false, false>(sc, px, py, pz, v, active ? seed * seed : -1.0, c, nullptr);
  if (active && v < seed) a.out_d[qi] = (float)v;
}

// The list's length is only known on the device: a fixed grid of wavefronts strides over it. The list
// holds near-surface queries from all over the scene, so a wavefront walks about one path per entry,
// and the slowest wavefront ends the launch: at most kScene64Lanes entries each (32M queries, 4,096
// spheres + 1,024 boxes + 8 meshes: 64 entries 0.98 ms, 32 0.79, 16 0.81), fewer while the list does
// not fill the grid twice (4M queries: 345 -> 280 us).
constexpr uint32_t kScene64Lanes = 32;
template <int KM, int NB>
__global__ __launch_bounds__(256) void scene64_kernel(const SceneDev sc, const QueryArgs a)
{
  const uint64_t n     = a.count_ptr ? (uint64_t)*a.count_ptr : a.n;
  const uint32_t lane  = __lane_id();
  const uint64_t waves = (uint64_t)gridDim.x * 4u;
  uint32_t       width = 1;
  while (width < kScene64Lanes && 2u * width * waves < n) width *= 2u;
  for (uint64_t w = uni(blockIdx.x * 4u + (threadIdx.x >> 6)); w * width < n; w += waves) {
    const uint64_t tid = lane < width ? w * width + lane : n; // n: inactive
    scene64_block<KM, NB>(sc, a, n, tid);
  }
}

template <int NB>
hipError_t launch32(const SceneDev& sc, const QueryArgs& a, SceneSlot* slots, bool count, hipStream_t s)
{
  const uint32_t blocks = (uint32_t)((a.n + 255) / 256);
  if (blocks == 0) return hipSuccess;
  if (count) hipLaunchKernelGGL((scene32_kernel<NB, true, false>), dim3(blocks), dim3(256), 0, s, sc, a, slots);
  else if (!slots) hipLaunchKernelGGL((scene32_kernel<NB, false, false>), dim3(blocks), dim3(256), 0, s, sc, a, slots);
  else {
    const HandOn& h = a.hand;
    if (a.seed_r || !h.slot_cap || !h.list || !h.keys || !h.items[0] || !h.items[1] || !h.counts) return hipErrorInvalidValue;
    const uint32_t g = std::clamp<uint32_t>(4u * blocks, 512u, 2048u);
    hipLaunchKernelGGL((scene32_kernel<NB, false, true>), dim3(blocks), dim3(256), 0, s, sc, a, slots);
    hipLaunchKernelGGL((scene_items_kernel<NB, 0>), dim3(g), dim3(256), 0, s, sc, a, slots);
    hipLaunchKernelGGL((scene_items_kernel<NB, 1>), dim3(g), dim3(256), 0, s, sc, a, slots);
    hipLaunchKernelGGL(scene_resolve_kernel, dim3(std::min(g, (h.slot_cap + 3u) / 4u)), dim3(256), 0, s, sc, a, slots);
  }
  return hipGetLastError();
}

template <int KM, int NB>
hipError_t launch64(const SceneDev& sc, const QueryArgs& a, hipStream_t s)
{
  const uint32_t blocks = (uint32_t)std::min<uint64_t>((a.n + 3) / 4, 2048u);
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL((scene64_kernel<KM, NB>), dim3(blocks), dim3(256), 0, s, sc, a);
  return hipGetLastError();
}

} // namespace

hipError_t launch_scene32(const SceneDev& sc, int banks, const QueryArgs& a, SceneSlot* slots, bool count, hipStream_t s)
{
  if (banks <= 1) return launch32<1>(sc, a, slots, count, s);
  if (banks == 2) return launch32<2>(sc, a, slots, count, s);
  return launch32<4>(sc, a, slots, count, s);
}

hipError_t launch_scene64(const SceneDev& sc, int KM, int banks, const QueryArgs& a, hipStream_t s)
{
  if (KM == 4) {
    if (banks <= 1) return launch64<4, 1>(sc, a, s);
    if (banks == 2) return launch64<4, 2>(sc, a, s);
    return launch64<4, 4>(sc, a, s);
  }
  if (banks <= 1) return launch64<8, 1>(sc, a, s);
  if (banks == 2) return launch64<8, 2>(sc, a, s);
  return launch64<8, 4>(sc, a, s);
}

} // namespace ebgpu
