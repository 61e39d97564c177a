// k-nearest-neighbour queries on point clouds, gfx950: PointCloudBVH::closestPoint(s) and
// nearestNeighbor(s) / allNearestNeighbors (Source/EBGeometry_PointCloudBVH.hpp:115-161,
// PointCloudBVHImplem.hpp:235-470), batched.
//
// The packet traversal of the mesh kernel with a point leaf: one query per lane, the 64 lanes of
// a wavefront walk the K-wide tree together (wave-uniform VGPR-lane stack, node records and leaf
// points read with scalar loads), a child is pushed when some lane's box distance^2 is below its
// bound, and each lane keeps its k best (d^2, cloud index) in registers, sorted, new entries after
// equal ones (the reference's strict-< insertion). The bound is the k-th best d^2 (+inf until k
// points are held). Self queries (the cloud's own points, in leaf order, so packets are spatially
// coherent) exclude the point's own index.
#include "kernels.hpp"
#include "traverse_dev.hpp"

#include <hip/hip_runtime.h>

namespace ebgpu {

namespace {

using namespace dev;

// A lane's k best entries, sorted, at the end of the arrays: the KMAX - k entries before them hold
// -inf, which nothing is below, so the bound is d[KMAX - 1] for every k and an insertion costs four
// instructions per entry (compare, median, two selects). With the entries at the start (five per
// entry, and a select chain for the k-th) 500,000 queries for 8 of 200,000 points took 372 us in
// this kernel, now 309.
template <int KMAX>
struct KBest
{
  float    d[KMAX];
  uint32_t id[KMAX];

  __device__ __forceinline__ void init(uint32_t k)
  {
#pragma unroll
    for (int i = 0; i < KMAX; i++) {
      d[i]  = (uint32_t)i + k < (uint32_t)KMAX ? -INFINITY : INFINITY;
      id[i] = kInvalid;
    }
  }
  // sorted insert (nothing changes for x >= bound()); equal distances keep their order (the new entry goes after them)
  __device__ __forceinline__ void insert(float x, uint32_t xi)
  {
    bool below[KMAX];
#pragma unroll
    for (int i = 0; i < KMAX; i++) below[i] = x < d[i];
#pragma unroll
    for (int i = KMAX - 1; i > 0; i--) {
      d[i]       = __builtin_amdgcn_fmed3f(d[i - 1], x, d[i]);
      uint32_t t = below[i] ? xi : id[i];
      asm("" : "+v"(t)); // selects, not branches
      id[i] = below[i - 1] ? id[i - 1] : t;
    }
    d[0]  = below[0] ? x : d[0];
    id[0] = below[0] ? xi : id[0];
  }
  __device__ __forceinline__ float bound() const { return d[KMAX - 1]; }
  // keeps the entries in one set of registers through the walk's loop; left to itself the compiler
  // carries a second set and copies (85 registers and 5 wavefronts per SIMD for 8 entries, not 54 and 8)
  __device__ __forceinline__ void pin()
  {
#pragma unroll
    for (int i = 0; i < KMAX; i++) asm volatile("" : "+v"(d[i]), "+v"(id[i]));
  }
};

template <int K, int NB, int KMAX>
__device__ __forceinline__ void knn_walk(const CloudDev& c, float px, float py, float pz, bool active,
                                         uint32_t exclude, KBest<KMAX>& kb)
{
  // Insertions by the whole wavefront, or by the lanes that have one. 8-wide nodes fill the scalar
  // registers, and with 4 or 8 entries the masks of the whole wavefront's form spill them: 200,000
  // queries of 100,000 points took 501 (4), 606 (5) and 755 us (8 nearest) with it, 377, 460 and 599 by
  // lanes; the other way round 233 and 268 us for 1, 921 and 959 for 16.
  constexpr bool kWhole = K == 4 || KMAX == 1 || KMAX == 16;
  const Node<K>* __restrict__ nodes = static_cast<const Node<K>*>(c.nodes);
  LaneStack<NB>               st;
  st.init();
  const int lane = __lane_id();
  const int rep  = rep_lane(active ? 0.0f : -1.0f);
  int       top  = 0;
  st.put(top++, Entry{0u, 0u, c.root_lo[0], c.root_lo[1], c.root_lo[2], c.root_hi[0], c.root_hi[1], c.root_hi[2]});
  while (top > 0) {
    const Entry e = st.get(--top);
    kb.pin();
    // a box at the bound can hold no new entry (strict <), but a lane without k points yet has
    // bound +inf; inactive lanes have bound -1
    float bound = active ? kb.bound() : -1.0f;
    const bool need = box_d2<float>(px, py, pz, e.lx, e.ly, e.lz, e.hx, e.hy, e.hz) < bound;
    if (ballot(need) == 0) continue;
    if (e.cnt == 0u) {
      push_children<K, NB, float, false>(sload_record(nodes + uni(e.ref)), px, py, pz, bound, st, top, rep);
      if (top > 64 * NB) {
        if (lane == 0 && c.status) atomicOr(c.status, kStatusStackOverflow);
        top = 64 * NB;
      }
      continue;
    }
    const uint32_t first = uni(e.ref), cnt = uni(e.cnt);
    for (uint32_t c0 = 0; c0 < cnt; c0 += 8) {
      // eight points (x, y, z, cloud index) per scalar round trip; the array is padded by 16
      const SWords<32> w = sload<32>(c.pts + 4 * (size_t)(first + c0));
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float    dx = px - __uint_as_float(w.w[4 * i]), dy = py - __uint_as_float(w.w[4 * i + 1]),
                       dz = pz - __uint_as_float(w.w[4 * i + 2]);
        const float    d2 = dx * dx + dy * dy + dz * dz;
        const uint32_t pi = w.w[4 * i + 3];
        const bool     in = d2 < bound && pi != exclude && c0 + i < cnt;
        if constexpr (kWhole) {
          if (ballot(in)) { // for the whole wavefront: the entries stay in their registers
            kb.insert(in ? d2 : INFINITY, pi); // +inf enters nowhere
            bound = active ? kb.bound() : -1.0f;
          }
        }
        else if (in) { // active lanes only
          kb.insert(d2, pi);
          bound = kb.bound();
        }
      }
    }
  }
}

template <int K, int NB, int KMAX>
__global__ __launch_bounds__(256) void knn_kernel(const CloudDev c, const KnnArgs a)
{
  const uint32_t blk = xcd_remap(blockIdx.x, gridDim.x);
  if ((uint64_t)blk * 256u >= a.n) return; // whole workgroup
  const uint64_t tid    = (uint64_t)blk * 256u + threadIdx.x;
  const bool     active = tid < a.n;
  float          px = 0.0f, py = 0.0f, pz = 0.0f;
  uint32_t       row = 0, exclude = kInvalid;
  if (active) {
    if (a.self) { // the cloud's own point at leaf position tid
      px      = __uint_as_float(c.pts[4 * tid]);
      py      = __uint_as_float(c.pts[4 * tid + 1]);
      pz      = __uint_as_float(c.pts[4 * tid + 2]);
      row     = c.pts[4 * tid + 3];
      exclude = row;
    }
    else {
      row = a.idx ? a.idx[tid] : (uint32_t)tid;
      px  = a.pts[3 * (size_t)row];
      py  = a.pts[3 * (size_t)row + 1];
      pz  = a.pts[3 * (size_t)row + 2];
    }
  }
  KBest<KMAX> kb;
  kb.init(a.k);
  knn_walk<K, NB, KMAX>(c, px, py, pz, active, exclude, kb);
  if (!active) return;
  const uint32_t skip = (uint32_t)KMAX - a.k;
#pragma unroll
  for (int i = 0; i < KMAX; i++) {
    if ((uint32_t)i >= skip) {
      a.out_idx[(size_t)row * a.k + (i - skip)] = kb.id[i];
      if (a.out_d2) a.out_d2[(size_t)row * a.k + (i - skip)] = kb.d[i];
    }
  }
}

template <int K, int NB, int KMAX>
hipError_t launch_k(const CloudDev& c, const KnnArgs& a, hipStream_t s)
{
  const uint32_t blocks = (uint32_t)((a.n + 255) / 256);
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL((knn_kernel<K, NB, KMAX>), dim3(blocks), dim3(256), 0, s, c, a);
  return hipGetLastError();
}

template <int K, int NB>
hipError_t launch_nb(const CloudDev& c, const KnnArgs& a, hipStream_t s)
{
  if (a.k <= 1) return launch_k<K, NB, 1>(c, a, s);
  if (a.k <= 4) return launch_k<K, NB, 4>(c, a, s);
  if (a.k <= 8) return launch_k<K, NB, 8>(c, a, s);
  return launch_k<K, NB, 16>(c, a, s);
}

} // namespace

hipError_t launch_knn(const CloudDev& c, int K, int banks, const KnnArgs& a, hipStream_t s)
{
  if (a.k < 1 || a.k > kKnnMax) return hipErrorInvalidValue;
  if (K == 4) {
    if (banks <= 1) return launch_nb<4, 1>(c, a, s);
    if (banks == 2) return launch_nb<4, 2>(c, a, s);
    return launch_nb<4, 4>(c, a, s);
  }
  if (banks <= 1) return launch_nb<8, 1>(c, a, s);
  if (banks == 2) return launch_nb<8, 2>(c, a, s);
  return launch_nb<8, 4>(c, a, s);
}

} // namespace ebgpu
