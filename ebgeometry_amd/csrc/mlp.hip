// Learned cull bound: fused MFMA inference, MFMA training GEMMs, Adam, sample generation.
//
// MFMA: v_mfma_f32_16x16x32_bf16 (gfx950). Operand layout per lane l (n = l % 16, g = l / 16):
//   A (16 x 32, M x K): row n, k = 8g .. 8g+7      B (32 x 16, K x N): column n, k = 8g .. 8g+7
//   D (16 x 16):        column n, rows 4g .. 4g+3
// The fused kernel computes h^T = W^T x^T per layer so that queries run along N. Layer L's
// accumulators hold, for query n, features 16t + 4g + e of output tile t; the next layer reads
// its B operand straight from them by taking the K order
//   phi(b, g, e) = 32b + (e < 4 ? 4g + e : 16 + 4g + e - 4)
// and storing the next weight matrix's A fragments in that same K order (no data movement).
#include "mlp.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

namespace ebgpu {

namespace {

typedef __bf16   bf16x8 __attribute__((ext_vector_type(8)));
typedef float    f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (v_cvt_pk_bf16_f32 on gfx950)
__device__ __forceinline__ uint16_t f2bf(float x) { return __builtin_bit_cast(uint16_t, (__bf16)x); }
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// relu(a), relu(b) as two BF16 in one word: one v_cvt_pk_bf16_f32 and one packed 16-bit integer
// max with 0 (a BF16 bit pattern is negative as an int16 exactly when the value is, -0 included)
typedef float  f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short  i16x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint32_t relu_pk_bf16(float a, float b)
{
  const bf16x2 h = __builtin_convertvector((f32x2){a, b}, bf16x2);
  const i16x2  r = __builtin_elementwise_max(__builtin_bit_cast(i16x2, h), (i16x2){0, 0});
  return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ f32x4 mfma(u16x8 a, u16x8 b, f32x4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}

// Fourier frequencies w_k = pi * 2^(0.4 k), k = 0..15, in revolutions per unit (w_k / 2 pi,
// float32-rounded): v_sin_f32 takes its argument in revolutions.
__constant__ float c_freq[kMlpFreqs];

struct MlpDev
{
  float           lo[3], sc[3], diag;
  const uint16_t* winfer;
  const float*    master;
};

__device__ __forceinline__ float feature(int f, float x0, float x1, float x2)
{
  if (f >= kMlpIn) return 0.0f;
  const int   c = f < 3 ? f : (f - 3) % 3;
  const float x = c == 0 ? x0 : (c == 1 ? x1 : x2);
  if (f < 3) return x;
  return __builtin_amdgcn_sinf(c_freq[(f - 3) / 3] * x);
}

// ------------------------------------------------------------------------------------------
// fused inference: one wavefront = kInferQT tiles of 16 queries, each weight fragment read from
// LDS once per kInferQT MFMAs; kInferWaves waves per workgroup.
// The BF16 weight fragments (116 KB) and the FP32 biases are copied once per workgroup into
// LDS and the workgroup then strides over query tiles (one workgroup per CU), so every A
// fragment comes from LDS instead of an L2 round trip per wavefront.
// ------------------------------------------------------------------------------------------

constexpr int kInferWaves = 12; // 3 per SIMD
constexpr int kInferQT    = 2;  // 16-query tiles per wavefront (32 queries; 148 VGPRs)
constexpr int kInferBias  = 4 * kMlpHidden; // b1..b4 in LDS

// Layer-1 K order of the fused kernel: K index 32 b + 8 g + e holds, for g < 3, the Fourier
// feature sin(w_j x_g) with j = 8 b + e, and for g = 3 the raw coordinate x_e (b = 0, e < 3)
// or zero padding (-1). A lane's frequencies are then compile-time constants and its coordinate
// is one select per query; features are bitwise those of the training kernel.
__host__ __device__ constexpr int infer_feature(int b, int g, int e)
{
  return g < 3 ? 3 + 3 * (8 * b + e) + g : (b == 0 && e < 3 ? e : -1);
}

__device__ __forceinline__ uint32_t pk_bf16(float a, float b)
{
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

// acc[q][t] += A(t, b) B_q(b) over the 8 NB fragments of one layer, K block b outermost so that
// consecutive MFMAs never chain on one accumulator; the A fragments stream from LDS through a
// ring of three registers, two loads ahead of the MFMAs that use them.
template <int NB>
__device__ __forceinline__ void layer_mma(const uint16_t* __restrict__ w, int lane, f32x4 (&acc)[kInferQT][8],
                                          const u16x8 (&bq)[kInferQT][4])
{
  constexpr int F = 8 * NB;
  auto frag = [&](int f) { return *reinterpret_cast<const u16x8*>(w + (((f % 8) * NB + f / 8) * 64 + lane) * 8); };
  u16x8 a[3];
  a[0] = frag(0);
  a[1] = frag(1);
#pragma unroll
  for (int f = 0; f < F; f++) {
    if (f + 2 < F) a[(f + 2) % 3] = frag(f + 2);
    const int t = f % 8, b = f / 8;
#pragma unroll
    for (int q = 0; q < kInferQT; q++) acc[q][t] = mfma(a[f % 3], bq[q][b], acc[q][t]);
  }
}

// One hidden layer (K = 128) from the previous layer's accumulators `prev` into `acc` (separate
// registers): K block b's B operands (relu'd BF16 of prev tiles 2b, 2b+1) are packed right
// before the MFMAs that read them, so that the packing of block b+1 can be scheduled under the
// MFMAs of block b.
__device__ __forceinline__ void dense_layer(const uint16_t* __restrict__ w, const float* __restrict__ bias, int lane,
                                            const f32x4 (&prev)[kInferQT][8], f32x4 (&acc)[kInferQT][8])
{
  const int g = lane >> 4;
#pragma unroll
  for (int t = 0; t < 8; t++) {
    const f32x4 bv = *reinterpret_cast<const f32x4*>(bias + 16 * t + 4 * g);
#pragma unroll
    for (int q = 0; q < kInferQT; q++) acc[q][t] = bv;
  }
  auto  frag = [&](int f) { return *reinterpret_cast<const u16x8*>(w + (((f % 8) * 4 + f / 8) * 64 + lane) * 8); };
  u16x8 a[3], bq[kInferQT];
  a[0] = frag(0);
  a[1] = frag(1);
#pragma unroll
  for (int f = 0; f < 32; f++) {
    const int t = f % 8, b = f / 8;
    if (t == 0) {
#pragma unroll
      for (int q = 0; q < kInferQT; q++) {
        const u32x4v v = {relu_pk_bf16(prev[q][2 * b][0], prev[q][2 * b][1]),
                          relu_pk_bf16(prev[q][2 * b][2], prev[q][2 * b][3]),
                          relu_pk_bf16(prev[q][2 * b + 1][0], prev[q][2 * b + 1][1]),
                          relu_pk_bf16(prev[q][2 * b + 1][2], prev[q][2 * b + 1][3])};
        bq[q]          = __builtin_bit_cast(u16x8, v);
      }
    }
    if (f + 2 < 32) a[(f + 2) % 3] = frag(f + 2);
#pragma unroll
    for (int q = 0; q < kInferQT; q++) acc[q][t] = mfma(a[f % 3], bq[q], acc[q][t]);
  }
}

__device__ __forceinline__ void infer_tile(const uint16_t* __restrict__ sw, const float* __restrict__ sb,
                                           const float* __restrict__ pts, const uint32_t* __restrict__ idx,
                                           uint64_t n, uint64_t base, const MlpDev& p, float b5, float scale,
                                           float offset, int seed_mode, float* __restrict__ out)
{
  const int lane = threadIdx.x & 63;
  const int nn = lane & 15, g = lane >> 4;

  u16x8    bq[kInferQT][4];
  uint32_t qid[kInferQT];
  bool     valid[kInferQT];
#pragma unroll
  for (int q = 0; q < kInferQT; q++) {
    const uint64_t i = base + q * 16 + nn;
    valid[q]         = i < n;
    qid[q]           = valid[q] ? (idx ? idx[i] : (uint32_t)i) : 0u;
    float x[3]       = {0.0f, 0.0f, 0.0f};
    if (valid[q])
      for (int c = 0; c < 3; c++) x[c] = (pts[3 * (size_t)qid[q] + c] - p.lo[c]) * p.sc[c] - 1.0f;
    // g = 3 lanes take 0 here, so their sin() terms are exactly the zero padding
    const float xg = g == 0 ? x[0] : (g == 1 ? x[1] : (g == 2 ? x[2] : 0.0f));
#pragma unroll
    for (int b = 0; b < 2; b++) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        v[e] = __builtin_amdgcn_sinf(c_freq[8 * b + e] * xg);
        if (b == 0 && e < 3) v[e] = g == 3 ? x[e] : v[e];
      }
      const u32x4v w = {pk_bf16(v[0], v[1]), pk_bf16(v[2], v[3]), pk_bf16(v[4], v[5]), pk_bf16(v[6], v[7])};
      bq[q][b] = __builtin_bit_cast(u16x8, w);
    }
  }

  // each layer's accumulators start from its bias (output rows 16 t + 4 g .. + 3 of this lane);
  // layers alternate between two accumulator sets
  f32x4 accA[kInferQT][8], accB[kInferQT][8];
#pragma unroll
  for (int t = 0; t < 8; t++) {
    const f32x4 bv = *reinterpret_cast<const f32x4*>(sb + 16 * t + 4 * g);
#pragma unroll
    for (int q = 0; q < kInferQT; q++) accA[q][t] = bv;
  }
  // layer 1 (K = 64)
  layer_mma<2>(sw + kBfW1, lane, accA, bq);
  // layers 2..4 (K = 128)
  dense_layer(sw + kBfW2, sb + 1 * kMlpHidden, lane, accA, accB);
  dense_layer(sw + kBfW3, sb + 2 * kMlpHidden, lane, accB, accA);
  dense_layer(sw + kBfW4, sb + 3 * kMlpHidden, lane, accA, accB);
  // output layer y = relu(h4) . w5 + b5 on MFMA: h4 rounded to BF16 as in training; rows 0..2 of
  // the W5 fragments are w5's three BF16 parts, so lanes g = 0 receive b5 + hi.h, mid.h, lo.h
  f32x4 y[kInferQT];
#pragma unroll
  for (int q = 0; q < kInferQT; q++) y[q] = (f32x4){b5, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int b = 0; b < 4; b++) {
    const u16x8 a = *reinterpret_cast<const u16x8*>(sw + kBfW5 + (b * 64 + lane) * 8);
#pragma unroll
    for (int q = 0; q < kInferQT; q++) {
      const u32x4v v = {relu_pk_bf16(accB[q][2 * b][0], accB[q][2 * b][1]),
                        relu_pk_bf16(accB[q][2 * b][2], accB[q][2 * b][3]),
                        relu_pk_bf16(accB[q][2 * b + 1][0], accB[q][2 * b + 1][1]),
                        relu_pk_bf16(accB[q][2 * b + 1][2], accB[q][2 * b + 1][3])};
      y[q]           = mfma(a, __builtin_bit_cast(u16x8, v), y[q]);
    }
  }
#pragma unroll
  for (int q = 0; q < kInferQT; q++) {
    if (g == 0 && valid[q]) {
      const float s = y[q][0] + y[q][1] + y[q][2];
      const float r = (expf(s) - kMlpLogC) * p.diag;
      out[qid[q]]   = seed_mode ? scale * fmaxf(r, 0.0f) + offset : r;
    }
  }
}

__global__ __launch_bounds__(64 * kInferWaves) void infer_kernel(const float* __restrict__ pts,
                                                                 const uint32_t* __restrict__ idx, uint64_t n, MlpDev p,
                                                                 float scale, float offset, int seed_mode,
                                                                 float* __restrict__ out)
{
  __shared__ __attribute__((aligned(16))) uint16_t sw[kBfInfer];
  __shared__ __attribute__((aligned(16))) float    sb[kInferBias];
  for (int i = 8 * threadIdx.x; i < kBfInfer; i += 8 * 64 * kInferWaves)
    *reinterpret_cast<u16x8*>(sw + i) = *reinterpret_cast<const u16x8*>(p.winfer + i);
  {
    const int bofs[4] = {kOffB1, kOffB2, kOffB3, kOffB4};
    for (int i = threadIdx.x; i < kInferBias; i += 64 * kInferWaves) sb[i] = p.master[bofs[i / kMlpHidden] + i % kMlpHidden];
  }
  __syncthreads();
  const float b5 = p.master[kOffB5];
  // every wavefront runs the same number of iterations of this loop shape (no barrier inside)
  const uint64_t per = 16u * kInferQT * kInferWaves;
  for (uint64_t tile = blockIdx.x; tile * per < n; tile += gridDim.x) {
    const uint64_t base = tile * per + 16u * kInferQT * (threadIdx.x >> 6);
    if (base < n) infer_tile(sw, sb, pts, idx, n, base, p, b5, scale, offset, seed_mode, out);
  }
}

// ------------------------------------------------------------------------------------------
// training: one launch for the loss and every gradient, one for the reduction and Adam
// ------------------------------------------------------------------------------------------

// A training step is 12 small products; as separate launches (25 a step, 16 x 16 tiles, operands
// through L2) it was bound by the launches: 262,144 samples in batches of 4,096, labelling included,
// took 13.7 ms, now 3.1 ms (a step: 30 us here, 6 us in the sums and Adam). Here a workgroup takes
// 64 rows through the whole network and back with every activation and delta in LDS (160 KB): only
// the points come in and the workgroup's gradient goes out. The gradient tiles stay in the
// accumulators over the workgroup's 64-row tiles, and each workgroup writes its own partial
// gradient, summed in a fixed order by the second launch: no atomics but the loss, so training is
// reproducible. What bounds it now is the chain of products and barriers of one tile (a step of
// 4,096 rows fills 64 workgroups).
// The operations and roundings are those of separate products: BF16 activations and deltas, FP32
// accumulation, FP32 biases, output layer and loss.
constexpr int kTrainWaves = 8;   // wave w owns output columns 16 w .. 16 w + 15 of every product
constexpr int kTrainLd    = kMlpHidden + 8; // LDS strides of row-major tiles (16-byte aligned, rows on
constexpr int kTrainLd0   = kMlpInPad + 8;  // shifted banks) ...
constexpr int kTrainLdT   = kTrainRows + 8; // ... and of tiles stored column by column

// Products along the network take a tile's rows as their operand, the weight gradients (in^T d) its
// columns: activations and deltas are stored both ways where both are read, so that every operand is
// one 16-byte read (gathering the columns from row-major tiles, 8 reads of 2 bytes each, a step of
// 4,096 rows took 39 us, now 30).
struct TrainLds
{
  uint16_t x0[kTrainRows * kTrainLd0], x0t[kMlpInPad * kTrainLdT];
  uint16_t r[3][kTrainRows * kTrainLd];   // rows of h1, h4, d2; of h2, d4; of h3, d3 (layers from 1)
  uint16_t ht[3][kMlpHidden * kTrainLdT]; // columns of h1, h2, h3
  uint16_t dt[2][kMlpHidden * kTrainLdT]; // columns of the deltas, in turn
  float    w5[kMlpHidden], g[kTrainRows];
};
static_assert(sizeof(TrainLds) <= 160 * 1024, "one training workgroup's LDS");

__device__ __forceinline__ u16x8 lds8(const uint16_t* p) { return *reinterpret_cast<const u16x8*>(p); }
__device__ __forceinline__ uint16_t relu_gate(uint16_t h, float x) { return f2bf((h == 0 || (h & 0x8000u)) ? 0.0f : x); }

// acc += in^T d over the tile's 64 rows: NT row tiles of in's columns, the wave's 16 columns of d
template <int NT>
__device__ __forceinline__ void train_wgrad(const uint16_t* in, const uint16_t* d, int wave, int nn, int g,
                                            f32x4 (&acc)[NT])
{
  const u16x8 b0 = lds8(d + (16 * wave + nn) * kTrainLdT + 8 * g);
  const u16x8 b1 = lds8(d + (16 * wave + nn) * kTrainLdT + 32 + 8 * g);
#pragma unroll
  for (int t = 0; t < NT; t++) {
    acc[t] = mfma(lds8(in + (16 * t + nn) * kTrainLdT + 8 * g), b0, acc[t]);
    acc[t] = mfma(lds8(in + (16 * t + nn) * kTrainLdT + 32 + 8 * g), b1, acc[t]);
    if (t & 1) __builtin_amdgcn_sched_barrier(0); // a few operands at a time: the registers hold the gradients
  }
}
// The wave's weight fragments of a layer of K inputs (K / 32 blocks), from the [out][in] copy.
template <int K>
__device__ __forceinline__ void train_weights(const uint16_t* w, int col, int g, u16x8 (&bf)[4])
{
#pragma unroll
  for (int b = 0; b < K / 32; b++) bf[b] = *reinterpret_cast<const u16x8*>(w + col * K + 32 * b + 8 * g);
}
// Rows 16 t .. 16 t + 15 of (in W) for the wave's 16 columns
template <int K>
__device__ __forceinline__ f32x4 train_rows(const uint16_t* in, int ld, int t, int nn, int g, const u16x8 (&bf)[4])
{
  f32x4 acc{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int b = 0; b < K / 32; b++) acc = mfma(lds8(in + (16 * t + nn) * ld + 32 * b + 8 * g), bf[b], acc);
  return acc;
}

// wt: the BF16 weights row-major [in][out]; wtt: the same transposed, [out][in] per layer (same
// offsets). part: kMaster floats per workgroup. Rows n and above of the last tile contribute nothing.
__global__ __launch_bounds__(64 * kTrainWaves) void train_kernel(const float* __restrict__ pts,
                                                                 const float* __restrict__ target, int n, MlpDev p,
                                                                 const uint16_t* __restrict__ wt,
                                                                 const uint16_t* __restrict__ wtt, float inv_diag,
                                                                 float inv_n, float under_weight,
                                                                 float* __restrict__ loss_sum, float* __restrict__ part)
{
  __shared__ __attribute__((aligned(16))) TrainLds S;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, nn = lane & 15,
            g   = lane >> 4;
  const int    col = 16 * wave + nn; // this lane's output column
  const float* mst = p.master;
  if (tid < kMlpHidden) S.w5[tid] = mst[kOffW5 + tid];
  const float b5 = mst[kOffB5];
  float       bias[4];
  {
    const int bo[4] = {kOffB1, kOffB2, kOffB3, kOffB4};
#pragma unroll
    for (int L = 0; L < 4; L++) bias[L] = mst[bo[L] + col];
  }
  f32x4 a1[4], a2[8], a3[8], a4[8]; // gradient tiles of W1..W4: rows 16 t + 4 g + e, column col
#pragma unroll
  for (int t = 0; t < 8; t++) {
    if (t < 4) a1[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    a2[t] = a3[t] = a4[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  // column sums: column tid / 4, a quarter of the rows each; db5, lsum: threads 0 mod 8
  float     db[4] = {0.0f, 0.0f, 0.0f, 0.0f}, dw5 = 0.0f, db5 = 0.0f, lsum = 0.0f;
  const int sc = tid >> 2, sq = tid & 3;
  const int wo[4] = {kBfW1, kBfW2, kBfW3, kBfW4};

  for (int row0 = blockIdx.x * kTrainRows; row0 < n; row0 += gridDim.x * kTrainRows) {
    // the weights are read again for each tile (kept across tiles they would take the registers that
    // hold the gradients), each layer's one layer ahead of its products
    const uint16_t *wl = wt, *wlt = wtt;
    asm volatile("" : "+s"(wl), "+s"(wlt));
    u16x8 bf[2][4];
    train_weights<kMlpInPad>(wlt + wo[0], col, g, bf[0]);
    const int r8 = tid >> 3, k8 = tid & 7; // 8 threads per row
    float     tgt = 0.0f;
    { // features: 8 per thread
      const int i = row0 + r8, f0 = k8 * 8;
      float     x[3] = {0.0f, 0.0f, 0.0f};
      if (i < n) {
        tgt = target[i];
        for (int c = 0; c < 3; c++) x[c] = (pts[3 * (size_t)i + c] - p.lo[c]) * p.sc[c] - 1.0f;
      }
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const uint16_t f = f2bf(feature(f0 + k, x[0], x[1], x[2]));
        S.x0[r8 * kTrainLd0 + f0 + k]    = f;
        S.x0t[(f0 + k) * kTrainLdT + r8] = f;
      }
    }
    __syncthreads();
    // forward: h = relu(in W + b)
#pragma unroll
    for (int L = 0; L < 4; L++) {
      if (L < 3) train_weights<kMlpHidden>(wlt + wo[L + 1], col, g, bf[(L + 1) & 1]);
      uint16_t* h = S.r[L == 3 ? 0 : L];
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const f32x4 acc = L == 0 ? train_rows<kMlpInPad>(S.x0, kTrainLd0, t, nn, g, bf[0])
                                 : train_rows<kMlpHidden>(S.r[L - 1], kTrainLd, t, nn, g, bf[L & 1]);
        u16x4       v;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          v[e] = f2bf(fmaxf(acc[e] + bias[L], 0.0f));
          h[(16 * t + 4 * g + e) * kTrainLd + col] = v[e];
        }
        if (L < 3) *reinterpret_cast<u16x4*>(&S.ht[L][col * kTrainLdT + 16 * t + 4 * g]) = v;
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
    }
    train_weights<kMlpHidden>(wl + wo[3], col, g, bf[1]);
    { // output layer and loss: 8 threads per row, columns 2 k8 + 16 j and the next
      const uint16_t* h = S.r[0] + r8 * kTrainLd + 2 * k8;
      uint32_t        hv[8];
      float           y = 0.0f;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        hv[j] = *reinterpret_cast<const uint32_t*>(h + 16 * j);
        y += bf2f((uint16_t)hv[j]) * S.w5[2 * k8 + 16 * j];
        y += bf2f((uint16_t)(hv[j] >> 16)) * S.w5[2 * k8 + 16 * j + 1];
      }
      for (int o = 1; o < 8; o <<= 1) y += __shfl_xor(y, o, 64);
      y += b5;
      float gi = 0.0f;
      if (row0 + r8 < n) {
        const float e = y - logf(fabsf(tgt) * inv_diag + kMlpLogC);
        const float w = e < 0.0f ? under_weight : 1.0f;
        gi            = 2.0f * w * e * inv_n;
        if (k8 == 0) lsum += w * e * e;
      }
      if (k8 == 0) {
        S.g[r8] = gi;
        db5 += gi;
      }
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int      c  = 2 * k8 + 16 * j;
        const uint16_t d0 = relu_gate((uint16_t)hv[j], gi * S.w5[c]), d1 = relu_gate((uint16_t)(hv[j] >> 16), gi * S.w5[c + 1]);
        *reinterpret_cast<uint32_t*>(&S.r[1][r8 * kTrainLd + c]) = d0 | (uint32_t)d1 << 16;
        S.dt[1][c * kTrainLdT + r8]                              = d0;
        S.dt[1][(c + 1) * kTrainLdT + r8]                        = d1;
      }
    }
    __syncthreads();
#pragma unroll 8
    for (int j = 0; j < kTrainRows / 4; j++) dw5 += bf2f(S.r[0][(4 * j + sq) * kTrainLd + sc]) * S.g[4 * j + sq];
    // hidden layers, last to first: the delta of layer L (from 0) has its columns in dt[L & 1], its
    // rows in r[1], r[2], r[0] for L = 3, 2, 1
#pragma unroll
    for (int L = 3; L >= 0; L--) {
      const uint16_t* d = S.dt[L & 1];
      if (L > 1) train_weights<kMlpHidden>(wl + wo[L - 1], col, g, bf[(L - 1) & 1]);
      {
        const u16x8 lo = lds8(d + sc * kTrainLdT + 16 * sq), hi = lds8(d + sc * kTrainLdT + 16 * sq + 8);
        float       s = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) s += bf2f(lo[e]);
#pragma unroll
        for (int e = 0; e < 8; e++) s += bf2f(hi[e]);
        db[L] += s;
      }
      if (L > 0) { // delta of the layer below: (d W^T) where its activation is positive
        const uint16_t* dr = S.r[L == 3 ? 1 : (L == 2 ? 2 : 0)];
        uint16_t*       o  = S.r[L == 3 ? 2 : 0];
#pragma unroll
        for (int t = 0; t < 4; t++) {
          const f32x4 acc = train_rows<kMlpHidden>(dr, kTrainLd, t, nn, g, bf[L & 1]);
          const u16x4 h   = *reinterpret_cast<const u16x4*>(&S.ht[L - 1][col * kTrainLdT + 16 * t + 4 * g]);
          u16x4       v;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            v[e] = relu_gate(h[e], acc[e]);
            if (L > 1) o[(16 * t + 4 * g + e) * kTrainLd + col] = v[e];
          }
          *reinterpret_cast<u16x4*>(&S.dt[(L - 1) & 1][col * kTrainLdT + 16 * t + 4 * g]) = v;
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (L == 3) train_wgrad<8>(S.ht[2], d, wave, nn, g, a4);
      else if (L == 2) train_wgrad<8>(S.ht[1], d, wave, nn, g, a3);
      else if (L == 1) train_wgrad<8>(S.ht[0], d, wave, nn, g, a2);
      else train_wgrad<4>(S.x0t, d, wave, nn, g, a1);
      __syncthreads();
    }
  }

  float* out = part + (size_t)blockIdx.x * kMaster;
#pragma unroll
  for (int t = 0; t < 8; t++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int r = (16 * t + 4 * g + e) * kMlpHidden + col;
      if (t < 4) out[kOffW1 + r] = a1[t][e];
      out[kOffW2 + r] = a2[t][e];
      out[kOffW3 + r] = a3[t][e];
      out[kOffW4 + r] = a4[t][e];
    }
  for (int o = 1; o < 4; o <<= 1) {
#pragma unroll
    for (int L = 0; L < 4; L++) db[L] += __shfl_xor(db[L], o, 64);
    dw5 += __shfl_xor(dw5, o, 64);
  }
  if (sq == 0) {
    const int bo[4] = {kOffB1, kOffB2, kOffB3, kOffB4};
#pragma unroll
    for (int L = 0; L < 4; L++) out[bo[L] + sc] = db[L];
    out[kOffW5 + sc] = dw5;
  }
  for (int o = 32; o > 0; o >>= 1) {
    lsum += __shfl_xor(lsum, o, 64);
    db5 += __shfl_xor(db5, o, 64);
  }
  if (lane == 0) S.g[wave] = db5; // after the last tile's barrier
  __syncthreads();
  if (tid == 0) {
    float s = 0.0f;
    for (int w = 0; w < kTrainWaves; w++) s += S.g[w];
    out[kOffB5] = s;
  }
  if (lane == 0 && lsum != 0.0f) atomicAdd(loss_sum, lsum);
}

// The step's gradient: the workgroups' partial gradients summed in order (grad), and with ADAM the
// update of the master weights and of both BF16 training copies.
template <bool ADAM>
__global__ __launch_bounds__(256) void train_update_kernel(const float* __restrict__ part, int parts,
                                                           float* __restrict__ grad, float* __restrict__ w,
                                                           float* __restrict__ m, float* __restrict__ v, float lr,
                                                           float bc1, float bc2, uint16_t* __restrict__ wt,
                                                           uint16_t* __restrict__ wtt)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= kMaster) return;
  float gi = 0.0f;
  int   b  = 0;
  for (; b + 8 <= parts; b += 8) { // eight loads in flight
    float x[8];
#pragma unroll
    for (int k = 0; k < 8; k++) x[k] = part[(size_t)(b + k) * kMaster + i];
#pragma unroll
    for (int k = 0; k < 8; k++) gi += x[k];
  }
  for (; b < parts; b++) gi += part[(size_t)b * kMaster + i];
  grad[i] = gi;
  if constexpr (ADAM) {
    const float mi = 0.9f * m[i] + 0.1f * gi;
    const float vi = 0.999f * v[i] + 0.001f * gi * gi;
    m[i]           = mi;
    v[i]           = vi;
    const float wi = w[i] - lr * (mi * bc1) / (sqrtf(vi * bc2) + 1e-8f);
    w[i]           = wi;
    const int mo[4] = {kOffW1, kOffW2, kOffW3, kOffW4}, wo[4] = {kBfW1, kBfW2, kBfW3, kBfW4};
#pragma unroll
    for (int L = 0; L < 4; L++) {
      const int K = L == 0 ? kMlpInPad : kMlpHidden, j = i - mo[L];
      if (j >= 0 && j < K * kMlpHidden) {
        const uint16_t q                                  = f2bf(wi);
        wt[wo[L] + j]                                     = q;
        wtt[wo[L] + (j % kMlpHidden) * K + j / kMlpHidden] = q;
      }
    }
  }
}

// BF16 copies: the training copies (row-major, and transposed per layer) and the permuted inference
// fragments.
__global__ __launch_bounds__(256) void sync_bf16_kernel(const float* __restrict__ master, uint16_t* __restrict__ wtrain,
                                                        uint16_t* __restrict__ wtrain_t, uint16_t* __restrict__ winfer)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= kBfInfer) return;
  // inference copy, fragment-major: A fragment (output tile t of 16 rows, K block b of 32) is
  // 64 lanes x 8 BF16 contiguous, lane = row + 16 g holding K elements 8 g .. 8 g + 7, so that a
  // wavefront's 16-byte LDS reads of one fragment fall on consecutive banks
  if (i >= kBfW5) {
    // output layer: row r < 3 of fragment b holds part r of w5 in the K order of layers 2..4
    const int j = i - kBfW5, e = j % 8, lane = (j / 8) % 64, b = j / 512, g = lane / 16, r = lane % 16;
    const int k = 32 * b + (e < 4 ? 4 * g + e : 16 + 4 * g + (e - 4));
    const float  w  = master[kOffW5 + k];
    const __bf16 hi = (__bf16)w;
    const float  r1 = w - (float)hi;
    const __bf16 mid = (__bf16)r1;
    const __bf16 lo  = (__bf16)(r1 - (float)mid);
    const __bf16 v   = r == 0 ? hi : (r == 1 ? mid : (r == 2 ? lo : (__bf16)0.0f));
    winfer[i]        = __builtin_bit_cast(uint16_t, v);
    return;
  }
  // training copy: same [in][out] layout as the master
  int src;
  if (i < kBfW2) src = kOffW1 + i;
  else if (i < kBfW3) src = kOffW2 + (i - kBfW2);
  else if (i < kBfW4) src = kOffW3 + (i - kBfW3);
  else src = kOffW4 + (i - kBfW4);
  wtrain[i] = f2bf(master[src]);
  const bool first = i < kBfW2;
  const int  base  = first ? kBfW1 : (i < kBfW3 ? kBfW2 : (i < kBfW4 ? kBfW3 : kBfW4));
  const int  moff  = first ? kOffW1 : (i < kBfW3 ? kOffW2 : (i < kBfW4 ? kOffW3 : kOffW4));
  const int  nb    = first ? kMlpInPad / 32 : kMlpHidden / 32;
  {
    const int K = first ? kMlpInPad : kMlpHidden, jj = i - base;
    wtrain_t[base + (jj % kMlpHidden) * K + jj / kMlpHidden] = wtrain[i];
  }
  const int  j = i - base, e = j % 8, lane = (j / 8) % 64, frag = j / 512;
  const int  t = frag / nb, b = frag % nb, g = lane / 16;
  const int  r = 16 * t + lane % 16;
  // K order: for layer 1 the feature order of infer_feature (padding -> zero weight); for
  // layers 2..4 the order in which the previous layer's accumulators sit in a lane (rows
  // 4 g .. 4 g + 3 of tiles 2b, 2b+1)
  const int k = first ? infer_feature(b, g, e) : 32 * b + (e < 4 ? 4 * g + e : 16 + 4 * g + (e - 4));
  winfer[i]   = k < 0 ? (uint16_t)0 : f2bf(master[moff + k * kMlpHidden + r]); // W^T[out r][in k]
}

// public order <-> master layout (W1 rows 51..63 are padding)
__global__ void grad_public_kernel(const float* __restrict__ g, float* __restrict__ out)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= kMlpParams) return;
  const int w1 = kMlpIn * kMlpHidden;
  out[i]       = i < w1 ? g[i] : g[i + (kMlpInPad - kMlpIn) * kMlpHidden];
}

// ------------------------------------------------------------------------------------------
// training samples
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ uint64_t mix64(uint64_t z)
{
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
__device__ __forceinline__ double u01(uint64_t key, uint64_t ctr)
{
  return (double)(mix64(key + ctr * 0x9E3779B97F4A7C15ull) >> 11) * (1.0 / 9007199254740992.0);
}

__global__ __launch_bounds__(256) void samples_kernel(MeshDev m, const float* __restrict__ cdf, uint32_t nt, float lo0,
                                                      float lo1, float lo2, float hi0, float hi1, float hi2,
                                                      float box_scale, float sigma, uint64_t key, uint64_t n,
                                                      float* __restrict__ out)
{
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const double lo[3] = {lo0, lo1, lo2}, hi[3] = {hi0, hi1, hi2};
  double       p[3];
  if ((i & 1u) == 0) { // even: uniform in the box; odd: near the surface (interleaved batches)
    for (int c = 0; c < 3; c++) {
      const double ctr = 0.5 * (lo[c] + hi[c]), h = 0.5 * box_scale * (hi[c] - lo[c]);
      p[c]             = ctr + h * (2.0 * u01(key, 8 * i + c) - 1.0);
    }
  }
  else {
    const float u = (float)u01(key, 8 * i);
    uint32_t    a = 0, b = nt - 1; // first t with cdf[t] > u
    while (a < b) {
      const uint32_t mid = (a + b) / 2;
      if (cdf[mid] > u) b = mid;
      else a = mid + 1;
    }
    const float*  x  = m.tripos + 12 * (size_t)a;
    const double* fn = m.fn64 + 4 * (size_t)a;
    const double  r1 = sqrt(u01(key, 8 * i + 1)), r2 = u01(key, 8 * i + 2);
    const double  u1 = u01(key, 8 * i + 3) + 1e-300, u2 = u01(key, 8 * i + 4);
    const double  z  = sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
    for (int c = 0; c < 3; c++)
      p[c] = (1.0 - r1) * x[c] + r1 * (1.0 - r2) * x[3 + c] + r1 * r2 * x[6 + c] + sigma * z * fn[c];
  }
  for (int c = 0; c < 3; c++) out[3 * i + c] = (float)p[c];
}

// Training samples of a union scene's bound: even i uniform in the training box, odd i uniform
// in the world box of a random primitive (the PrimRec bounding boxes) grown by sigma on each side.
__global__ __launch_bounds__(256) void scene_samples_kernel(const PrimRec* __restrict__ prims, uint32_t np, float lo0,
                                                            float lo1, float lo2, float hi0, float hi1, float hi2,
                                                            float box_scale, float sigma, uint64_t key, uint64_t n,
                                                            float* __restrict__ out)
{
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const double lo[3] = {lo0, lo1, lo2}, hi[3] = {hi0, hi1, hi2};
  double       p[3];
  if ((i & 1u) == 0) {
    for (int c = 0; c < 3; c++) {
      const double ctr = 0.5 * (lo[c] + hi[c]), h = 0.5 * box_scale * (hi[c] - lo[c]);
      p[c]             = ctr + h * (2.0 * u01(key, 8 * i + c) - 1.0);
    }
  }
  else {
    const uint32_t k  = min(np - 1, (uint32_t)(u01(key, 8 * i) * np));
    const float*   bv = prims[k].bv;
    for (int c = 0; c < 3; c++)
      p[c] = (double)bv[c] - sigma + ((double)bv[3 + c] - bv[c] + 2.0 * sigma) * u01(key, 8 * i + 1 + c);
  }
  for (int c = 0; c < 3; c++) out[3 * i + c] = (float)p[c];
}

MlpDev dev_of(const Mlp& m)
{
  MlpDev d;
  for (int c = 0; c < 3; c++) {
    d.lo[c] = m.lo[c];
    d.sc[c] = m.scale[c];
  }
  d.diag   = m.diag;
  d.winfer = m.winfer;
  d.master = m.master;
  return d;
}

hipError_t upload_freqs()
{
  static bool done = false;
  if (done) return hipSuccess;
  float f[kMlpFreqs];
  for (int k = 0; k < kMlpFreqs; k++) f[k] = (float)(0.5 * std::pow(2.0, 0.4 * k)); // pi 2^(0.4k) / (2 pi)
  hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_freq), f, sizeof(f));
  if (e == hipSuccess) done = true;
  return e;
}

} // namespace

Mlp::~Mlp()
{
  for (void* p : {(void*)master, (void*)grad, (void*)adam_m, (void*)adam_v, (void*)wtrain, (void*)wtrain_t, (void*)winfer})
    if (p) (void)hipFree(p);
}

MlpTrainBuffers::~MlpTrainBuffers()
{
  for (void* p : {(void*)part, (void*)loss})
    if (p) (void)hipFree(p);
}

hipError_t MlpTrainBuffers::ensure(int b)
{
  const int want = mlp_train_blocks(b);
  hipError_t e;
  if (!loss && (e = hipMalloc(&loss, sizeof(float) * 4)) != hipSuccess) return e;
  if (want <= parts) return hipSuccess;
  if (part) (void)hipFree(part);
  part  = nullptr;
  parts = 0;
  if ((e = hipMalloc(&part, sizeof(float) * kMaster * want)) != hipSuccess) return e;
  parts = want;
  return hipSuccess;
}

hipError_t mlp_alloc(Mlp& m)
{
  hipError_t e = upload_freqs();
  if (e != hipSuccess) return e;
  if (m.master) return hipSuccess;
  if ((e = hipMalloc(&m.master, sizeof(float) * kMaster)) != hipSuccess) return e;
  if ((e = hipMalloc(&m.grad, sizeof(float) * kMaster)) != hipSuccess) return e;
  if ((e = hipMalloc(&m.adam_m, sizeof(float) * kMaster)) != hipSuccess) return e;
  if ((e = hipMalloc(&m.adam_v, sizeof(float) * kMaster)) != hipSuccess) return e;
  if ((e = hipMalloc(&m.wtrain, sizeof(uint16_t) * kBfTotal)) != hipSuccess) return e;
  if ((e = hipMalloc(&m.wtrain_t, sizeof(uint16_t) * kBfTotal)) != hipSuccess) return e;
  if ((e = hipMalloc(&m.winfer, sizeof(uint16_t) * kBfInfer)) != hipSuccess) return e;
  if ((e = hipMemset(m.grad, 0, sizeof(float) * kMaster)) != hipSuccess) return e;
  return hipSuccess;
}

static void public_to_master(const float* pub, std::vector<float>& mst)
{
  mst.assign(kMaster, 0.0f);
  const int w1 = kMlpIn * kMlpHidden;
  for (int i = 0; i < kMlpParams; i++) mst[i < w1 ? i : i + (kMlpInPad - kMlpIn) * kMlpHidden] = pub[i];
}

hipError_t mlp_set_params_host(Mlp& m, const float* params)
{
  hipError_t e = mlp_alloc(m);
  if (e != hipSuccess) return e;
  std::vector<float> mst;
  public_to_master(params, mst);
  if ((e = hipMemcpy(m.master, mst.data(), sizeof(float) * kMaster, hipMemcpyHostToDevice)) != hipSuccess) return e;
  if ((e = hipMemset(m.adam_m, 0, sizeof(float) * kMaster)) != hipSuccess) return e;
  if ((e = hipMemset(m.adam_v, 0, sizeof(float) * kMaster)) != hipSuccess) return e;
  m.step = 0;
  if ((e = mlp_sync_bf16(m, nullptr)) != hipSuccess) return e;
  return hipDeviceSynchronize();
}

hipError_t mlp_get_params_host(const Mlp& m, float* params)
{
  if (!m.master) return hipErrorInvalidValue;
  std::vector<float> mst(kMaster);
  hipError_t         e = hipMemcpy(mst.data(), m.master, sizeof(float) * kMaster, hipMemcpyDeviceToHost);
  if (e != hipSuccess) return e;
  const int w1 = kMlpIn * kMlpHidden;
  for (int i = 0; i < kMlpParams; i++) params[i] = mst[i < w1 ? i : i + (kMlpInPad - kMlpIn) * kMlpHidden];
  return hipSuccess;
}

hipError_t mlp_init(Mlp& m, uint64_t seed)
{
  // He-uniform weights from SplitMix64, zero biases
  std::vector<float> pub(kMlpParams, 0.0f);
  uint64_t           s    = seed ? seed : 1;
  auto               next = [&s]() {
    s += 0x9E3779B97F4A7C15ull;
    uint64_t z = s;
    z          = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z          = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (double)(z >> 11) * (1.0 / 9007199254740992.0);
  };
  int o = 0;
  auto fill = [&](int fan_in, int count) {
    const double a = std::sqrt(6.0 / fan_in);
    for (int i = 0; i < count; i++) pub[o + i] = float((2.0 * next() - 1.0) * a);
    o += count;
  };
  fill(kMlpIn, kMlpIn * kMlpHidden);
  o += kMlpHidden;
  for (int l = 0; l < 3; l++) {
    fill(kMlpHidden, kMlpHidden * kMlpHidden);
    o += kMlpHidden;
  }
  // small output layer: the first predictions sit near log(0.05) for every point
  const double a5 = 0.01 * std::sqrt(6.0 / kMlpHidden);
  for (int i = 0; i < kMlpHidden; i++) pub[o + i] = float((2.0 * next() - 1.0) * a5);
  o += kMlpHidden;
  pub[o] = float(std::log(0.05));
  return mlp_set_params_host(m, pub.data());
}

hipError_t mlp_sync_bf16(Mlp& m, hipStream_t s)
{
  hipLaunchKernelGGL(sync_bf16_kernel, dim3((kBfInfer + 255) / 256), dim3(256), 0, s, m.master, m.wtrain, m.wtrain_t,
                     m.winfer);
  return hipGetLastError();
}

hipError_t mlp_forward(const Mlp& m, const float* pts, const uint32_t* idx, uint64_t n, bool seed_mode, float scale,
                       float offset, float* out, hipStream_t s)
{
  if (n == 0) return hipSuccess;
  // one workgroup per CU (the weights take 112 KB of the CU's LDS)
  static int cus = 0;
  if (!cus) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      cus = 256;
  }
  const uint64_t tiles  = (n + 16 * kInferQT * kInferWaves - 1) / (16 * kInferQT * kInferWaves);
  const uint32_t blocks = (uint32_t)std::min<uint64_t>(tiles, (uint64_t)cus);
  hipLaunchKernelGGL(infer_kernel, dim3(blocks), dim3(64 * kInferWaves), 0, s, pts, idx, n, dev_of(m), scale, offset,
                     seed_mode ? 1 : 0, out);
  return hipGetLastError();
}

// Enqueue the loss and the partial gradients of a step over n rows of `samples`; returns the partial
// gradients' number in *parts. Weights, biases and gradients have fixed sizes; what depends on n is checked.
static hipError_t train_launch(Mlp& m, MlpTrainBuffers& tb, const float* pts, const float* target, uint64_t samples, int n,
                               hipStream_t s, int* parts, std::string* why)
{
  if (!check_train_step(n, samples, uint64_t(tb.parts), why)) return hipErrorInvalidValue;
  *parts = mlp_train_blocks(n);
  hipLaunchKernelGGL(train_kernel, dim3(*parts), dim3(64 * kTrainWaves), 0, s, pts, target, n, dev_of(m), m.wtrain,
                     m.wtrain_t, 1.0f / m.diag, 1.0f / (float)n, m.under_weight, tb.loss, tb.part);
  return hipGetLastError();
}

hipError_t mlp_loss_grad(Mlp& m, MlpTrainBuffers& tb, const float* pts, const float* target, int n, hipStream_t s,
                         std::string* why)
{
  hipError_t e     = tb.ensure(n);
  int        parts = 0;
  if (e != hipSuccess || (e = train_launch(m, tb, pts, target, uint64_t(n), n, s, &parts, why)) != hipSuccess)
    return e;
  hipLaunchKernelGGL(train_update_kernel<false>, dim3((kMaster + 255) / 256), dim3(256), 0, s, tb.part, parts, m.grad,
                     nullptr, nullptr, nullptr, 0.0f, 0.0f, 0.0f, nullptr, nullptr);
  return hipGetLastError();
}

hipError_t mlp_step(Mlp& m, MlpTrainBuffers& tb, const float* pts, const float* target, uint64_t samples, int n, float lr,
                    hipStream_t s, std::string* why)
{
  int        parts = 0;
  hipError_t e     = train_launch(m, tb, pts, target, samples, n, s, &parts, why);
  if (e != hipSuccess) return e;
  m.step++;
  const float bc1 = 1.0f / (1.0f - std::pow(0.9f, (float)m.step));
  const float bc2 = 1.0f / (1.0f - std::pow(0.999f, (float)m.step));
  hipLaunchKernelGGL(train_update_kernel<true>, dim3((kMaster + 255) / 256), dim3(256), 0, s, tb.part, parts, m.grad,
                     m.master, m.adam_m, m.adam_v, lr, bc1, bc2, m.wtrain, m.wtrain_t);
  return hipGetLastError();
}

hipError_t mlp_grad_public(const Mlp& m, float* out, hipStream_t s)
{
  hipLaunchKernelGGL(grad_public_kernel, dim3((kMlpParams + 255) / 256), dim3(256), 0, s, m.grad, out);
  return hipGetLastError();
}

hipError_t mlp_samples(const MeshDev& dev, const float* cdf, uint32_t nt, const float* lo, const float* hi,
                       float box_scale, float sigma, uint64_t seed, uint64_t n, float* pts, hipStream_t s)
{
  if (n == 0) return hipSuccess;
  uint64_t key = seed * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E019ull;
  hipLaunchKernelGGL(samples_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, dev, cdf, nt, lo[0], lo[1],
                     lo[2], hi[0], hi[1], hi[2], box_scale, sigma, key, n, pts);
  return hipGetLastError();
}

hipError_t mlp_scene_samples(const PrimRec* prims, uint32_t num_prims, const float* lo, const float* hi,
                             float box_scale, float sigma, uint64_t seed, uint64_t n, float* pts, hipStream_t s)
{
  if (n == 0 || num_prims == 0) return hipSuccess;
  uint64_t key = seed * 0x9E3779B97F4A7C15ull + 0x2545F4914F6CDD1Dull;
  hipLaunchKernelGGL(scene_samples_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, prims, num_prims, lo[0],
                     lo[1], lo[2], hi[0], hi[1], hi[2], box_scale, sigma, key, n, pts);
  return hipGetLastError();
}

hipError_t mlp_fit(Mlp& m, MlpTrainBuffers& tb, const float* pts, const float* dist, uint64_t n, int epochs, int batch,
                   float lr0, hipStream_t s, float* last_loss, std::string* why)
{
  hipError_t e = tb.ensure(batch);
  if (e != hipSuccess) return e;
  // Adam with a cosine learning-rate decay to 5% over all steps
  const uint64_t spe   = train_steps(n, batch);
  const double   total = double(spe) * epochs;
  float          last  = 0.0f;
  for (int ep = 0; ep < epochs; ep++) {
    if ((e = hipMemsetAsync(tb.loss, 0, sizeof(float), s)) != hipSuccess) return e;
    for (uint64_t k = 0; k < spe; k++) {
      const TrainStep t  = train_step(n, batch, k);
      const float     lr = float(lr0 * (0.05 + 0.95 * 0.5 * (1.0 + std::cos(M_PI * double(ep * spe + k) / total))));
      if ((e = mlp_step(m, tb, pts + 3 * t.first, dist + t.first, n - t.first, t.rows, lr, s, why)) != hipSuccess) return e;
    }
    float sum = 0.0f;
    if ((e = hipMemcpyAsync(&sum, tb.loss, sizeof(float), hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
    if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
    last = sum / float(n);
  }
  if (last_loss) *last_loss = last;
  return mlp_sync_bf16(m, s); // the inference copy of the trained weights
}

} // namespace ebgpu
