// Small device utilities used by the query pipeline. Counters are cleared with a kernel (not
// hipMemsetAsync) so that a captured hipGraph replays them correctly.
#include "kernels.hpp"

#include <hip/hip_runtime.h>

namespace ebgpu {

namespace {

__global__ void fill_u32_kernel(uint32_t* p, uint64_t n, uint32_t v)
{
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = v;
}

// v[i] <- map[v[i]] for entries inside the map (kInvalid and other out-of-map values kept)
__global__ void map_u32_kernel(uint32_t* v, uint64_t n, const uint32_t* map, uint32_t nmap)
{
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) {
    const uint32_t x = v[i];
    if (x < nmap) v[i] = map[x];
  }
}

__global__ void add_counts_kernel(unsigned long long* work, const uint32_t* a, const uint32_t* b)
{
  if (threadIdx.x == 0) {
    if (a) work[2] += *a;
    if (b) work[3] += *b;
  }
}

// FP64 points rounded to FP32 (round to nearest even, as the host's (float) cast); FP32 results
// widened to FP64.
__global__ void f64_to_f32_kernel(const double* __restrict__ in, float* __restrict__ out, uint64_t n)
{
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = __double2float_rn(in[i]);
}

__global__ void f32_to_f64_kernel(const float* __restrict__ in, double* __restrict__ out, uint64_t n)
{
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = (double)in[i];
}

// 64 points (4 x 4 x 4) in each cell of g.dims cells of size g.spacing, cell by cell
__global__ void cell_points_kernel(GridSpec g, float* __restrict__ out)
{
  const uint64_t p = (uint64_t)blockIdx.x * 256 + threadIdx.x, c = p >> 6;
  const uint32_t l = (uint32_t)p & 63u;
  if (c >= g.dims[0] * g.dims[1] * g.dims[2]) return;
  const uint64_t i = c % g.dims[0], r = c / g.dims[0], j = r % g.dims[1], k = r / g.dims[1];
  out[3 * p]       = (float)(g.origin[0] + ((double)i + ((l & 3u) + 0.5) / 4) * g.spacing[0]);
  out[3 * p + 1]   = (float)(g.origin[1] + ((double)j + (((l >> 2) & 3u) + 0.5) / 4) * g.spacing[1]);
  out[3 * p + 2]   = (float)(g.origin[2] + ((double)k + ((l >> 4) + 0.5) / 4) * g.spacing[2]);
}

// Lattice points of a box of cells or nodes (x fastest, then y, then z: the layout of an AMReX
// or Chombo FAB): point (i, j, k) = origin + (i, j, k) * spacing, each coordinate a separately
// rounded FP64 product and sum, then rounded to FP32 (round to nearest even).
__global__ void grid_points_kernel(GridSpec g, float* __restrict__ out)
{
  const uint64_t n = g.dims[0] * g.dims[1] * g.dims[2];
  const uint64_t p = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= n) return;
  const uint64_t i = p % g.dims[0], r = p / g.dims[0];
  const uint64_t j = r % g.dims[1], k = r / g.dims[1];
  out[3 * p]       = __double2float_rn(__dadd_rn(g.origin[0], __dmul_rn((double)i, g.spacing[0])));
  out[3 * p + 1]   = __double2float_rn(__dadd_rn(g.origin[1], __dmul_rn((double)j, g.spacing[1])));
  out[3 * p + 2]   = __double2float_rn(__dadd_rn(g.origin[2], __dmul_rn((double)k, g.spacing[2])));
}

// Reductions over a workgroup of B threads, every thread getting the result.
template <int B, class Op>
__device__ __forceinline__ double block_reduce(double v, Op op)
{
  for (int o = 32; o > 0; o >>= 1) v = op(v, __shfl_xor(v, o, 64));
  if constexpr (B > 64) {
    __shared__ double sh[B / 64];
    __syncthreads();
    if ((threadIdx.x & 63u) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    v = sh[0];
    for (int i = 1; i < B / 64; i++) v = op(v, sh[i]);
  }
  return v;
}
template <int B>
__device__ __forceinline__ double block_sum(double v)
{
  return block_reduce<B>(v, [](double a, double b) { return a + b; });
}
template <int B>
__device__ __forceinline__ double block_max(double v)
{
  return block_reduce<B>(v, [](double a, double b) { return fmax(a, b); });
}

// The cylinder of a range of triangles (one workgroup per listed child slot): axis along the
// area-weighted normal, centre by extents along the axis and two directions across it, then moved
// towards the farthest corner a few times (keeping the best), radius and half-height measured
// from the centre and axis as rounded to FP32. The FP32 test (disc_lanes) rounds its own
// quantities by up to 2^-21 of the record's size and of the cull radius, squared; the record's
// part is covered here: R^2 + 2^-18 (R + t)^2, t + 2^-19 (R + t), rounded up. Everything depends
// on the set of triangles only, up to the FP64 rounding of the normal's sum. A range whose normal
// cancels has no axis: v[6] = -1, its node keeps the boxes.
template <int B>
__global__ __launch_bounds__(B) void walk_disc_kernel(const float* __restrict__ tripos, const uint32_t* __restrict__ range,
                                                      const uint32_t* __restrict__ list, double scale,
                                                      float* __restrict__ discs)
{
  const uint32_t slot = list[blockIdx.x], f = range[2 * (size_t)slot], l = range[2 * (size_t)slot + 1];
  float*         out  = discs + 8 * (size_t)slot;
  double         N[3] = {0.0, 0.0, 0.0}, A = 0.0;
  for (uint32_t t = f + threadIdx.x; t < l; t += B) {
    const float* x = tripos + 12 * (size_t)t;
    double       a[3], b[3];
    for (int c = 0; c < 3; c++) {
      a[c] = ((double)x[3 + c] - x[c]) * scale;
      b[c] = ((double)x[6 + c] - x[c]) * scale;
    }
    const double cx = a[1] * b[2] - a[2] * b[1], cy = a[2] * b[0] - a[0] * b[2], cz = a[0] * b[1] - a[1] * b[0];
    N[0] += cx;
    N[1] += cy;
    N[2] += cz;
    A += sqrt(cx * cx + cy * cy + cz * cz);
  }
  for (int c = 0; c < 3; c++) N[c] = block_sum<B>(N[c]);
  A               = block_sum<B>(A);
  const double nl = sqrt(N[0] * N[0] + N[1] * N[1] + N[2] * N[2]);
  if (!(nl > 0.3 * A)) { // whole workgroup
    if (threadIdx.x == 0) out[6] = -1.0f;
    return;
  }
  float  nr[3];
  double n[3], u[3], w[3];
  for (int c = 0; c < 3; c++) n[c] = nr[c] = (float)(N[c] / nl);
  {
    const int m = fabs(n[0]) < 0.7 ? 0 : 1; // a coordinate axis away from n
    double    q = 0.0;
    for (int c = 0; c < 3; c++) u[c] = (c == m ? 1.0 : 0.0) - n[m] * n[c] / (n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
    for (int c = 0; c < 3; c++) q += u[c] * u[c];
    for (int c = 0; c < 3; c++) u[c] /= sqrt(q);
    const double nn = sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
    w[0] = (n[1] * u[2] - n[2] * u[1]) / nn;
    w[1] = (n[2] * u[0] - n[0] * u[2]) / nn;
    w[2] = (n[0] * u[1] - n[1] * u[0]) / nn;
  }
  // extents along u, w and the axis (as -min, max)
  double e[6];
  for (int i = 0; i < 6; i++) e[i] = -INFINITY;
  for (uint32_t t = f + threadIdx.x; t < l; t += B) {
    const float* x = tripos + 12 * (size_t)t;
    for (int v = 0; v < 3; v++) {
      const double px = x[3 * v] * scale, py = x[3 * v + 1] * scale, pz = x[3 * v + 2] * scale;
      const double pu = u[0] * px + u[1] * py + u[2] * pz, pw = w[0] * px + w[1] * py + w[2] * pz,
                   ph = n[0] * px + n[1] * py + n[2] * pz;
      e[0] = fmax(e[0], -pu), e[1] = fmax(e[1], pu);
      e[2] = fmax(e[2], -pw), e[3] = fmax(e[3], pw);
      e[4] = fmax(e[4], -ph), e[5] = fmax(e[5], ph);
    }
  }
  for (int i = 0; i < 6; i++) e[i] = block_max<B>(e[i]);
  double       cu = 0.5 * (e[1] - e[0]), cw = 0.5 * (e[3] - e[2]), bu = cu, bw = cw, best = INFINITY;
  const double ch = 0.5 * (e[5] - e[4]) / (n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
  for (int it = 0; it < 8; it++) {
    double far = -1.0, fu = 0.0, fw = 0.0; // the farthest corner in the plane (ties: largest pu, then pw)
    for (uint32_t t = f + threadIdx.x; t < l; t += B) {
      const float* x = tripos + 12 * (size_t)t;
      for (int v = 0; v < 3; v++) {
        const double px = x[3 * v] * scale, py = x[3 * v + 1] * scale, pz = x[3 * v + 2] * scale;
        const double pu = u[0] * px + u[1] * py + u[2] * pz, pw = w[0] * px + w[1] * py + w[2] * pz;
        const double d  = (pu - cu) * (pu - cu) + (pw - cw) * (pw - cw);
        if (d > far || (d == far && (pu > fu || (pu == fu && pw > fw)))) {
          far = d;
          fu  = pu;
          fw  = pw;
        }
      }
    }
    const double m  = block_max<B>(far);
    const double mu = block_max<B>(far == m ? fu : -INFINITY);
    const double mw = block_max<B>(far == m && fu == mu ? fw : -INFINITY);
    if (m < best) {
      best = m;
      bu   = cu;
      bw   = cw;
    }
    cu += (mu - cu) * (0.5 / (it + 2));
    cw += (mw - cw) * (0.5 / (it + 2));
  }
  float cr[3];
  for (int c = 0; c < 3; c++) cr[c] = (float)(bu * u[c] + bw * w[c] + ch * n[c]);
  double t2 = 0.0, r2 = 0.0;
  for (uint32_t t = f + threadIdx.x; t < l; t += B) {
    const float* x = tripos + 12 * (size_t)t;
    for (int v = 0; v < 3; v++) {
      const double sx = x[3 * v] * scale - cr[0], sy = x[3 * v + 1] * scale - cr[1], sz = x[3 * v + 2] * scale - cr[2];
      const double pd = n[0] * sx + n[1] * sy + n[2] * sz;
      t2              = fmax(t2, fabs(pd));
      r2              = fmax(r2, sx * sx + sy * sy + sz * sz - pd * pd);
    }
  }
  t2 = block_max<B>(t2);
  r2 = block_max<B>(r2);
  if (threadIdx.x == 0) {
    const double s = sqrt(r2) + t2;
    for (int c = 0; c < 3; c++) {
      out[c]     = cr[c];
      out[3 + c] = nr[c];
    }
    out[6] = __double2float_ru(4.0 * (r2 + 0x1p-18 * s * s) * (1.0 + 1e-12));
    out[7] = __double2float_ru((t2 + 0x1p-19 * s) * (1.0 + 1e-12));
  }
}

// Per node: its children's cylinders in place of their boxes where every child has one that is
// flat (t < 0.4 R: a patch bent further than that is left to its box, whose distance also orders
// the children better: 40 against 60 nodes per packet on the 327,680-face displaced sphere) and
// the cylinders, grown by a quarter of their radius, hold less volume than the boxes grown alike
// (axis-aligned flat patches keep their boxes).
__global__ __launch_bounds__(256) void walk_node_kernel(WalkNode* __restrict__ nodes, uint32_t num_nodes,
                                                        const float* __restrict__ discs)
{
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= num_nodes) return;
  WalkNode& nd = nodes[i];
  double    vd = 0.0, vb = 0.0;
  for (int k = 0; k < 4; k++) {
    if (nd.cnt[k] == kInvalid) continue;
    const float* d = discs + 8 * ((size_t)4 * i + k);
    if (!(d[6] >= 0.0f)) return;
    const double R = 0.5 * sqrt((double)d[6]), t = d[7], g = 0.25 * R;
    if (!(t < 0.4 * R)) return;
    vd += 2.0 * (t + g) * M_PI * (R + g) * (R + g);
    vb += ((double)nd.v[k][3] - nd.v[k][0] + 2 * g) * ((double)nd.v[k][4] - nd.v[k][1] + 2 * g) *
          ((double)nd.v[k][5] - nd.v[k][2] + 2 * g);
  }
  if (!(vd < vb)) return;
  for (int k = 0; k < 4; k++) {
    if (nd.cnt[k] == kInvalid) continue;
    for (int j = 0; j < 8; j++) nd.v[k][j] = discs[8 * ((size_t)4 * i + k) + j];
    nd.cnt[k] &= ~kBoxChild;
  }
}

// The in-plane frame record of each triangle (FrameRec), in FP64 from the FP32 vertices: the
// longest edge becomes A -> B (a zero-length longest edge, a point triangle, takes the x axis),
// ey is the unit part of C - A normal to ex (when C lies on the line AB, any unit vector normal
// to ex: then c = 0 and no point is inside the face), ez = ex x ey. The edge parameters of a
// zero-length edge are 0, so that edge's closest point is its start. Beside it the triangle's
// culling disc: the smallest circle of its plane that holds it (on the longest edge when the angle
// at C is not acute, else through the corners), radius and the corners' distance from the disc's
// plane measured from the centre and normal as rounded to FP32; the largest such distance of the
// mesh goes to *off (float bits, zero on entry). All times `scale`.
__global__ __launch_bounds__(256) void frame_kernel(const float* __restrict__ tripos, uint64_t nt, double scale,
                                                    FrameRec* __restrict__ out, TriDisc* __restrict__ disc,
                                                    uint32_t* __restrict__ off)
{
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= nt) return;
  const float* x = tripos + 12 * i;
  double       P[3][3];
  for (int v = 0; v < 3; v++)
    for (int c = 0; c < 3; c++) P[v][c] = x[3 * v + c] * scale;
  double L[3];
  for (int j = 0; j < 3; j++) {
    const int k = j == 2 ? 0 : j + 1;
    L[j]        = 0.0;
    for (int c = 0; c < 3; c++) L[j] += (P[k][c] - P[j][c]) * (P[k][c] - P[j][c]);
  }
  int j = 0;
  if (L[1] > L[j]) j = 1;
  if (L[2] > L[j]) j = 2;
  const double* A = P[j];
  const double* B = P[j == 2 ? 0 : j + 1];
  const double* C = P[j == 0 ? 2 : j - 1];
  const double  a = sqrt(L[j]);
  double        ex[3] = {1.0, 0.0, 0.0}, ey[3], ez[3];
  if (a > 0.0)
    for (int c = 0; c < 3; c++) ex[c] = (B[c] - A[c]) / a;
  double b = 0.0;
  for (int c = 0; c < 3; c++) b += (C[c] - A[c]) * ex[c];
  double rr[3], cc = 0.0;
  for (int c = 0; c < 3; c++) {
    rr[c] = (C[c] - A[c]) - b * ex[c];
    cc += rr[c] * rr[c];
  }
  cc = sqrt(cc);
  if (!(cc > 0.0)) {
    // the coordinate axis least aligned with ex, made normal to it
    int m = 0;
    if (fabs(ex[1]) < fabs(ex[m])) m = 1;
    if (fabs(ex[2]) < fabs(ex[m])) m = 2;
    double nr = 0.0;
    for (int c = 0; c < 3; c++) {
      rr[c] = (c == m ? 1.0 : 0.0) - ex[m] * ex[c];
      nr += rr[c] * rr[c];
    }
    nr = sqrt(nr);
    for (int c = 0; c < 3; c++) ey[c] = rr[c] / nr;
    cc = 0.0;
  }
  else
    for (int c = 0; c < 3; c++) ey[c] = rr[c] / cc;
  ez[0] = ex[1] * ey[2] - ex[2] * ey[1];
  ez[1] = ex[2] * ey[0] - ex[0] * ey[2];
  ez[2] = ex[0] * ey[1] - ex[1] * ey[0];
  const double L1 = (b - a) * (b - a) + cc * cc, L2 = b * b + cc * cc;
  FrameRec     r{};
  for (int c = 0; c < 3; c++) {
    r.o[c]  = (float)A[c];
    r.ex[c] = (float)ex[c];
    r.ey[c] = (float)ey[c];
    r.ez[c] = (float)ez[c];
  }
  r.a   = (float)a;
  r.b   = (float)b;
  r.c   = (float)cc;
  r.bma = (float)(b - a);
  r.ca  = (float)(cc * a);
  r.k1u = L1 > 0.0 ? (float)((b - a) / L1) : 0.0f;
  r.k1v = L1 > 0.0 ? (float)(cc / L1) : 0.0f;
  r.k1c = L1 > 0.0 ? (float)(-a * (b - a) / L1) : 0.0f;
  r.k2u = L2 > 0.0 ? (float)(b / L2) : 0.0f;
  r.k2v = L2 > 0.0 ? (float)(cc / L2) : 0.0f;
  out[i] = r;

  double ou = 0.5 * a, ov = 0.0; // circle centre in the frame
  if ((b - ou) * (b - ou) + cc * cc > ou * ou) ov = 0.5 * (b * b - a * b + cc * cc) / cc;
  TriDisc d;
  for (int c = 0; c < 3; c++) {
    d.c[c] = (float)(A[c] + ou * ex[c] + ov * ey[c]);
    d.n[c] = (float)ez[c];
  }
  double t2 = 0.0, r2 = 0.0;
  for (int v = 0; v < 3; v++) {
    const double sx = P[v][0] - d.c[0], sy = P[v][1] - d.c[1], sz = P[v][2] - d.c[2];
    const double pd = (double)d.n[0] * sx + (double)d.n[1] * sy + (double)d.n[2] * sz;
    t2              = fmax(t2, fabs(pd));
    r2              = fmax(r2, sx * sx + sy * sy + sz * sz - pd * pd);
  }
  const double g = (r2 + 0x1p-18 * (sqrt(r2) + t2) * (sqrt(r2) + t2)) * (1.0 + 1e-12);
  d.r2x4  = __double2float_ru(4.0 * g);
  d.nr2   = -__double2float_ru(g);
  disc[i] = d;
  // the distance from the disc's plane, and the part of the test's own rounding that scales with
  // the record's size (as in walk_disc_kernel)
  atomicMax(off, __float_as_uint(__double2float_ru((t2 + 0x1p-19 * (sqrt(r2) + t2)) * (1.0 + 1e-12))));
}

} // namespace

hipError_t launch_frames(const float* tripos, uint64_t nt, float scale, FrameRec* out, TriDisc* disc, uint32_t* off,
                         hipStream_t s)
{
  if (nt == 0) return hipSuccess;
  hipLaunchKernelGGL(frame_kernel, dim3((uint32_t)((nt + 255) / 256)), dim3(256), 0, s, tripos, nt, (double)scale, out,
                     disc, off);
  return hipGetLastError();
}

hipError_t launch_walk_nodes(const float* tripos, const uint32_t* range, const uint32_t* small, uint32_t num_small,
                             const uint32_t* large, uint32_t num_large, float scale, float* discs, WalkNode* nodes,
                             uint32_t num_nodes, hipStream_t s)
{
  if (num_small)
    hipLaunchKernelGGL(walk_disc_kernel<64>, dim3(num_small), dim3(64), 0, s, tripos, range, small, (double)scale, discs);
  if (num_large)
    hipLaunchKernelGGL(walk_disc_kernel<1024>, dim3(num_large), dim3(1024), 0, s, tripos, range, large, (double)scale,
                       discs);
  if (num_nodes)
    hipLaunchKernelGGL(walk_node_kernel, dim3((num_nodes + 255) / 256), dim3(256), 0, s, nodes, num_nodes, discs);
  return hipGetLastError();
}

hipError_t launch_grid_points(const GridSpec& g, float* out, hipStream_t s)
{
  const uint64_t n = g.dims[0] * g.dims[1] * g.dims[2];
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(grid_points_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, g, out);
  return hipGetLastError();
}

hipError_t launch_cell_points(const GridSpec& g, float* out, hipStream_t s)
{
  const uint64_t n = 64 * g.dims[0] * g.dims[1] * g.dims[2];
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(cell_points_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, g, out);
  return hipGetLastError();
}

hipError_t launch_f64_to_f32(const double* in, float* out, uint64_t n, hipStream_t s)
{
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(f64_to_f32_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, in, out, n);
  return hipGetLastError();
}

hipError_t launch_f32_to_f64(const float* in, double* out, uint64_t n, hipStream_t s)
{
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(f32_to_f64_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, in, out, n);
  return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t s)
{
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(fill_u32_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

hipError_t launch_map_u32(uint32_t* v, uint64_t n, const uint32_t* map, uint32_t nmap, hipStream_t s)
{
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(map_u32_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, v, n, map, nmap);
  return hipGetLastError();
}

hipError_t launch_add_counts(unsigned long long* work, const uint32_t* recheck, const uint32_t* fallback, hipStream_t s)
{
  hipLaunchKernelGGL(add_counts_kernel, dim3(1), dim3(64), 0, s, work, recheck, fallback);
  return hipGetLastError();
}

} // namespace ebgpu
