// Learned GJK warm start for gfx950.
//
// A 39-128-128-128-4 multilayer perceptron with GELU (erf form) maps the
// relative pose of a pair plus a 16-float descriptor of each shape to an
// initial GJK search direction (3, in shape a's frame) and a signed-distance
// estimate (1).  Its output only seeds GJK through the reference's guess hook
// (GJKSolver::gjk_guess, include/fcl/narrowphase/detail/gjk_solver.h:140-163);
// the exact algorithm still decides every result.
//
// Every product runs on the MFMA units as BF16 x BF16 -> FP32
// (v_mfma_f32_32x32x16_bf16), each wavefront carrying 32 rows through the
// whole network with its activations in registers: inference and training
// write no activation to memory.  Training keeps FP32 master weights with
// Adam; BF16 images of the weights, in the order the products read them,
// are refreshed after each update.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "ctx.h"

namespace mfcl {

#define MFCL_LDS __attribute__((address_space(3)))

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
// four floats of a caller's array, which is aligned to one (a 16-byte load all the same)
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kBlk = 256;

// GELU from the normal distribution's tail q(t) = Phi(-t), t = |x|: log2 q is
// smooth, and takes a polynomial of degree 10 (least squares, reweighted
// towards the largest error in q).  No branch: erff's two ranges both ran for
// every value (the lanes differ), and took most of the inference kernel.
// Largest error over [-12, 12] against 64 bits: GELU 2.6e-7 (with erff
// 4.5e-7), its derivative 1.3e-7 (1.4e-7).
__device__ __forceinline__ float normalTail(float x) {
  const float t = fabsf(x);
  float p = -1.339073474e-08f;
  p = __builtin_fmaf(p, t, 5.026773238e-07f);
  p = __builtin_fmaf(p, t, -7.691206520e-06f);
  p = __builtin_fmaf(p, t, 6.081214087e-05f);
  p = __builtin_fmaf(p, t, -2.368241694e-04f);
  p = __builtin_fmaf(p, t, -6.996445154e-05f);
  p = __builtin_fmaf(p, t, 7.014930714e-03f);
  p = __builtin_fmaf(p, t, -5.247886106e-02f);
  p = __builtin_fmaf(p, t, -4.592103362e-01f);
  p = __builtin_fmaf(p, t, -1.151105285e+00f);
  p = __builtin_fmaf(p, t, -1.0f);
  return __builtin_amdgcn_exp2f(p);
}
// x Phi(x) = max(x, 0) - |x| q; NaN for an infinite x (with erff for -inf alone:
// the next layer's sums of mixed signs are NaN from either)
__device__ __forceinline__ float geluF(float x, float q) { return __builtin_fmaf(-fabsf(x), q, fmaxf(x, 0.f)); }
__device__ __forceinline__ float geluF(float x) { return geluF(x, normalTail(x)); }
// GELU's derivative Phi(x) + x phi(x)
__device__ __forceinline__ float geluGradF(float x, float q) {
  return __builtin_fmaf(x * 0.39894228040143268f, __builtin_amdgcn_exp2f(x * x * -0.72134752044448170f),
                        x > 0.f ? 1.f - q : q);
}
// The 16 accumulators of unit tile t start from the units' biases.
__device__ __forceinline__ f32x16 biasTile(const float* bias, int t, int h) {
  f32x16 acc;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 b = *reinterpret_cast<const float4*>(bias + 32 * t + 8 * q + 4 * h);
    acc[4 * q] = b.x;
    acc[4 * q + 1] = b.y;
    acc[4 * q + 2] = b.z;
    acc[4 * q + 3] = b.w;
  }
  return acc;
}

// ---------------------------------------------------------------- features
// Per pair: relative translation of b in a's frame (3), relative rotation
// quaternion (4, w >= 0), descriptors of a and b (16 + 16); columns 39..63
// are zero.
__global__ void __launch_bounds__(kBlk) featureKernel(const uint32_t* pa, const uint32_t* pb, const float* posea,
                                                      const float* poseb, const float* desc, uint32_t n_shapes,
                                                      uint64_t n, float* xf) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float f[kMlpInPad];
  for (int k = 0; k < kMlpInPad; ++k) f[k] = 0.f;
  if (pa[i] < n_shapes && pb[i] < n_shapes) {
    const float* A = posea + 7 * i;
    const float* B = poseb + 7 * i;
    float qa[4] = {A[3], A[4], A[5], A[6]}, qb[4] = {B[3], B[4], B[5], B[6]};
    const float na = rsqrtf(qa[0] * qa[0] + qa[1] * qa[1] + qa[2] * qa[2] + qa[3] * qa[3]);
    const float nb = rsqrtf(qb[0] * qb[0] + qb[1] * qb[1] + qb[2] * qb[2] + qb[3] * qb[3]);
    for (int k = 0; k < 4; ++k) { qa[k] *= na; qb[k] *= nb; }
    // R_a^T (t_b - t_a): rotate by the conjugate of q_a
    const float dx = B[0] - A[0], dy = B[1] - A[1], dz = B[2] - A[2];
    const float w = qa[0], x = -qa[1], y = -qa[2], z = -qa[3];
    const float tx = 2.f * (y * dz - z * dy), ty = 2.f * (z * dx - x * dz), tz = 2.f * (x * dy - y * dx);
    f[0] = dx + w * tx + (y * tz - z * ty);
    f[1] = dy + w * ty + (z * tx - x * tz);
    f[2] = dz + w * tz + (x * ty - y * tx);
    // q_a^* q_b
    float rw = w * qb[0] - x * qb[1] - y * qb[2] - z * qb[3];
    float rx = w * qb[1] + x * qb[0] + y * qb[3] - z * qb[2];
    float ry = w * qb[2] - x * qb[3] + y * qb[0] + z * qb[1];
    float rz = w * qb[3] + x * qb[2] - y * qb[1] + z * qb[0];
    if (rw < 0) { rw = -rw; rx = -rx; ry = -ry; rz = -rz; }
    f[3] = rw; f[4] = rx; f[5] = ry; f[6] = rz;
    const float* da = desc + 16 * static_cast<size_t>(pa[i]);
    const float* db = desc + 16 * static_cast<size_t>(pb[i]);
    for (int k = 0; k < 16; ++k) { f[7 + k] = da[k]; f[23 + k] = db[k]; }
  }
  for (int k = 0; k < kMlpInPad; ++k) xf[i * kMlpInPad + k] = f[k];
}

__global__ void fillKernel(float* p, uint64_t n, float v) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// --------------------------------------------------------- weight images
// Formulation: C = W . X^T (rows = units, columns = rows of the batch), so a
// layer's accumulator tile holds, in lane l, batch row l % 32 and the 16
// units 8 (r / 4) + 4 (l / 32) + r % 4 of the tile; the next layer takes
// those registers directly as its B operand (8 per K step) by contracting
// over the units in that order -- the packed weights are laid out with the
// same permutation of K, so no transpose through LDS is needed.
//
// Packed image (bf16x8 per lane): [layer][out tile][K step][lane], with
//   element i of lane l = W[32 t + l % 32][k(j, l / 32, i)],
//   layer 1: k = 16 j + 8 h + i (features in natural order),
//   layers 2-4: k = 32 (j / 2) + 16 (j % 2) + 8 (i / 4) + 4 h + i % 4;
// then, for the backward products (C = W^T . dZ), the same of the
// transposed layers 4 (one K step: four output units), 3 and 2:
//   element i of lane l = W[k(j, l / 32, i)][32 t + l % 32].
constexpr int kPackL1 = 4 * 4, kPackL2 = 4 * 8, kPackL3 = 4 * 8, kPackL4 = 1 * 8;  // (tile, K step) blocks
constexpr int kPackFwd = kPackL1 + kPackL2 + kPackL3 + kPackL4;
constexpr int kPackT4 = 4 * 1, kPackT3 = 4 * 8, kPackT2 = 4 * 8;
constexpr int kPackBlocks = kPackFwd + kPackT4 + kPackT3 + kPackT2;
constexpr int kPackFwdBytes = kPackFwd * 64 * 16;
constexpr int kPackBytes = kPackBlocks * 64 * 16;
constexpr int kPackBiasFloats = 3 * kHid + kMlpOutPad;

__device__ __forceinline__ int permK(int j, int h, int i) { return 32 * (j / 2) + 16 * (j % 2) + 8 * (i / 4) + 4 * h + (i % 4); }

__global__ void packKernel(const float* P, __bf16* pack, float* bias) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;  // one (block, lane, element)
  if (idx < kPackBlocks * 64 * 8) {
    const int e = idx % 8, l = (idx / 8) % 64, b = idx / (8 * 64);
    const int h = l / 32, m = l % 32;
    float v;
    if (b < kPackL1) {
      const int t = b / 4, j = b % 4;
      v = P[kOffW1 + (32 * t + m) * kMlpInPad + 16 * j + 8 * h + e];
    } else if (b < kPackL1 + kPackL2) {
      const int q = b - kPackL1, t = q / 8, j = q % 8;
      v = P[kOffW2 + (32 * t + m) * kHid + permK(j, h, e)];
    } else if (b < kPackL1 + kPackL2 + kPackL3) {
      const int q = b - kPackL1 - kPackL2, t = q / 8, j = q % 8;
      v = P[kOffW3 + (32 * t + m) * kHid + permK(j, h, e)];
    } else if (b < kPackFwd) {
      const int j = b - kPackL1 - kPackL2 - kPackL3;
      v = P[kOffW4 + m * kHid + permK(j, h, e)];
    } else if (b < kPackFwd + kPackT4) {
      const int t = b - kPackFwd;
      v = P[kOffW4 + permK(0, h, e) * kHid + 32 * t + m];
    } else if (b < kPackFwd + kPackT4 + kPackT3) {
      const int q = b - kPackFwd - kPackT4, t = q / 8, j = q % 8;
      v = P[kOffW3 + permK(j, h, e) * kHid + 32 * t + m];
    } else {
      const int q = b - kPackFwd - kPackT4 - kPackT3, t = q / 8, j = q % 8;
      v = P[kOffW2 + permK(j, h, e) * kHid + 32 * t + m];
    }
    pack[idx] = static_cast<__bf16>(v);
  }
  if (idx < kPackBiasFloats) {
    const int off = idx < kHid ? kOffB1 + idx
                  : idx < 2 * kHid ? kOffB2 + idx - kHid
                  : idx < 3 * kHid ? kOffB3 + idx - 2 * kHid : kOffB4 + idx - 3 * kHid;
    bias[idx] = P[off];
  }
}

__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// ------------------------------------------------------- fused inference
// Features, the four layers and the normalisation in one kernel: weights
// live in LDS (copied once per block from the packed image), and each
// wavefront carries 32 pairs through the network.

// one hidden layer: 4 output tiles, KS K steps, B operands in x[KS]
template <int KS>
__device__ __forceinline__ void denseGelu(const MFCL_LDS bf16x8* W, const bf16x8* x, const float* bias, int lane,
                                          bf16x8* out) {
  const int h = lane >> 5;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    f32x16 acc = biasTile(bias, t, h);
#pragma unroll
    for (int j = 0; j < KS; ++j) acc = mfma(W[(t * KS + j) * 64 + lane], x[j], acc);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bf16x8 o;
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = static_cast<__bf16>(geluF(acc[8 * s + i]));
      out[2 * t + s] = o;
    }
    // keep the scheduler from overlapping the tiles (register pressure)
    __builtin_amdgcn_sched_barrier(0);
  }
}
// Layers 1-4 on the feature operands x0: outputs 0..3 of row lane % 32 are
// registers 0..3 of the lanes below 32 (bias not added).
__device__ __forceinline__ f32x16 network(const MFCL_LDS bf16x8* W, const float* bias, const bf16x8* x0, int lane) {
  const MFCL_LDS bf16x8* W2 = W + kPackL1 * 64;
  const MFCL_LDS bf16x8* W3 = W2 + kPackL2 * 64;
  const MFCL_LDS bf16x8* W4 = W3 + kPackL3 * 64;
  bf16x8 a1[8], a2[8];
  denseGelu<4>(W, x0, bias, lane, a1);
  denseGelu<8>(W2, a1, bias + kHid, lane, a2);
  denseGelu<8>(W3, a2, bias + 2 * kHid, lane, a1);
  f32x16 acc = {};
#pragma unroll
  for (int j = 0; j < 8; ++j) acc = mfma(W4[j * 64 + lane], a1[j], acc);
  return acc;
}
// The weights into the block's LDS (dynamic, kPackFwdBytes + biases).
__device__ __forceinline__ void loadWeights(uint4* lds, const uint4* pack, const float* bias_g, const float*& bias) {
  for (int k = threadIdx.x; k < kPackFwdBytes / 16; k += blockDim.x) lds[k] = pack[k];
  float* b = reinterpret_cast<float*>(lds + kPackFwdBytes / 16);
  for (int k = threadIdx.x; k < kPackBiasFloats; k += blockDim.x) b[k] = bias_g[k];
  bias = b;
  __syncthreads();
}
// Feature row i (zeros from n on) as B operands: lanes h = 0 / 1 hold
// columns 16 j + 0..7 / 16 j + 8..15.
__device__ __forceinline__ void featureOperands(const float* xf, uint64_t i, uint64_t n, int h, bf16x8* x0) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f32x4u u = {0, 0, 0, 0}, w = u;
    if (i < n) {
      const f32x4u* f = reinterpret_cast<const f32x4u*>(xf + i * kMlpInPad + 16 * j + 8 * h);
      u = f[0];
      w = f[1];
    }
    const float v[8] = {u.x, u.y, u.z, u.w, w.x, w.y, w.z, w.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) x0[j][e] = static_cast<__bf16>(v[e]);
  }
}

// The forward pass on feature rows.
__global__ void __launch_bounds__(512) mlpForwardFused(const float* xf, uint64_t n, const uint4* pack_g,
                                                       const float* bias_g, float* y4) {
  extern __shared__ __align__(16) uint4 lds_pack[];
  const float* bias;
  loadWeights(lds_pack, pack_g, bias_g, bias);
  const MFCL_LDS bf16x8* W = (const MFCL_LDS bf16x8*)(lds_pack);
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const uint64_t ntiles = (n + 31) / 32;
  const uint64_t wave = (static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
  const uint64_t nwaves = (static_cast<uint64_t>(gridDim.x) * blockDim.x) >> 6;
  for (uint64_t tile = wave; tile < ntiles; tile += nwaves) {
    const uint64_t i = tile * 32 + (lane & 31);
    bf16x8 x0[4];
    featureOperands(xf, i, n, h, x0);
    const f32x16 acc = network(W, bias, x0, lane);
    if (h == 0 && i < n) {
      const float* b4 = bias + 3 * kHid;
      // rows of 4 floats; the caller's pointer need not be 16-byte aligned
      for (int k = 0; k < 4; ++k) y4[4 * i + k] = acc[k] + b4[k];
    }
  }
}

// BLK threads per block share the block's LDS copy of the weights (one
// block per CU): more wavefronts per block hide the feature loads and the
// MFMA chains behind each other, within BLK's register budget.
template <int BLK>
__global__ void __launch_bounds__(BLK) mlpGuessFused(const uint32_t* pa, const uint32_t* pb, const float* posea,
                                                      const float* poseb, const float* desc, uint32_t n_shapes,
                                                      uint64_t n, const uint4* pack_g, const float* bias_g, int policy,
                                                      float* guess3, float* dist) {
  extern __shared__ __align__(16) uint4 lds_pack[];
  const float* bias;
  loadWeights(lds_pack, pack_g, bias_g, bias);
  const MFCL_LDS bf16x8* W = (const MFCL_LDS bf16x8*)(lds_pack);
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const uint64_t ntiles = (n + 31) / 32;
  const uint64_t wave = (static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
  const uint64_t nwaves = (static_cast<uint64_t>(gridDim.x) * blockDim.x) >> 6;
  for (uint64_t tile = wave; tile < ntiles; tile += nwaves) {
    const uint64_t i = tile * 32 + (lane & 31);
    // features (the same formulas as featureKernel); lanes h = 0 / 1 keep
    // columns 16 j + 0..7 / 16 j + 8..15
    float t0 = 0, t1 = 0, t2 = 0, r0 = 0, r1 = 0, r2 = 0, r3 = 0;
    float4 da[4] = {}, db[4] = {};
    if (i < n && pa[i] < n_shapes && pb[i] < n_shapes) {
      const float* A = posea + 7 * i;
      const float* B = poseb + 7 * i;
      float qa[4] = {A[3], A[4], A[5], A[6]}, qb[4] = {B[3], B[4], B[5], B[6]};
      const float na = rsqrtf(qa[0] * qa[0] + qa[1] * qa[1] + qa[2] * qa[2] + qa[3] * qa[3]);
      const float nb = rsqrtf(qb[0] * qb[0] + qb[1] * qb[1] + qb[2] * qb[2] + qb[3] * qb[3]);
#pragma unroll
      for (int k = 0; k < 4; ++k) { qa[k] *= na; qb[k] *= nb; }
      const float dx = B[0] - A[0], dy = B[1] - A[1], dz = B[2] - A[2];
      const float w = qa[0], x = -qa[1], y = -qa[2], z = -qa[3];
      const float tx = 2.f * (y * dz - z * dy), ty = 2.f * (z * dx - x * dz), tz = 2.f * (x * dy - y * dx);
      t0 = dx + w * tx + (y * tz - z * ty);
      t1 = dy + w * ty + (z * tx - x * tz);
      t2 = dz + w * tz + (x * ty - y * tx);
      r0 = w * qb[0] - x * qb[1] - y * qb[2] - z * qb[3];
      r1 = w * qb[1] + x * qb[0] + y * qb[3] - z * qb[2];
      r2 = w * qb[2] - x * qb[3] + y * qb[0] + z * qb[1];
      r3 = w * qb[3] + x * qb[2] - y * qb[1] + z * qb[0];
      if (r0 < 0) { r0 = -r0; r1 = -r1; r2 = -r2; r3 = -r3; }
      const float4* pda = reinterpret_cast<const float4*>(desc + 16 * static_cast<size_t>(pa[i]));
      const float4* pdb = reinterpret_cast<const float4*>(desc + 16 * static_cast<size_t>(pb[i]));
#pragma unroll
      for (int q = 0; q < 4; ++q) { da[q] = pda[q]; db[q] = pdb[q]; }
    }
    // feature k: 0-2 t, 3-6 r, 7-22 da, 23-38 db, 39-63 zero
    auto feat = [&](int k) -> float {
      if (k < 3) return k == 0 ? t0 : (k == 1 ? t1 : t2);
      if (k < 7) return k == 3 ? r0 : (k == 4 ? r1 : (k == 5 ? r2 : r3));
      if (k < 23) { const float4 v = da[(k - 7) / 4]; const int c = (k - 7) % 4; return c == 0 ? v.x : (c == 1 ? v.y : (c == 2 ? v.z : v.w)); }
      if (k < 39) { const float4 v = db[(k - 23) / 4]; const int c = (k - 23) % 4; return c == 0 ? v.x : (c == 1 ? v.y : (c == 2 ? v.z : v.w)); }
      return 0.f;
    };
    bf16x8 x0[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) x0[j][e] = static_cast<__bf16>(h ? feat(16 * j + 8 + e) : feat(16 * j + e));
    const f32x16 acc = network(W, bias, x0, lane);
    // outputs 0..3 of pair lane % 32 are rows 0..3: registers 0..3 of the lanes with h = 0
    if (h == 0 && i < n) {
      const float* b4 = bias + 3 * kHid;
      const float y0 = acc[0] + b4[0], y1 = acc[1] + b4[1], y2 = acc[2] + b4[2], y3 = acc[3] + b4[3];
      const float nn = sqrtf(y0 * y0 + y1 * y1 + y2 * y2);
      float g0 = 1.f, g1 = 0.f, g2 = 0.f;
      if (nn > 1e-20f && !(policy == 1 && y3 < 0.f)) { g0 = y0 / nn; g1 = y1 / nn; g2 = y2 / nn; }
      guess3[3 * i] = g0;
      guess3[3 * i + 1] = g1;
      guess3[3 * i + 2] = g2;
      if (dist) dist[i] = y3;
    }
  }
}

// ------------------------------------------------------- fused training
// Forward, loss, backward and the weight gradients of 128 rows per block
// and step, 32 rows per wavefront, in one persistent kernel (one block of
// four wavefronts per CU).  The layered kernels this replaces wrote and read
// every activation, its transpose and its pre-activation (5.4 KB a row) and
// took 0.86 ms of a 65,536-row step's 0.92 ms, against 17 GFLOP of products
// (7 us of the MFMA units).
//
// Forward as in inference, GELU's derivative kept in FP32.  A
// weight gradient dW = dZ . H^T contracts over the rows, so its operands
// need the rows of one unit in one lane: the transpose of an activation tile
// is a product with the identity (exact: one term per sum), whose
// accumulators, rounded back to the BF16 values they are, go to LDS as
// operands.  All four wavefronts' operands (128 rows) are then contracted by
// the wavefront that owns the output tiles: wavefront w keeps the gradient
// rows 32 w .. 32 w + 31 of layers 1-3 and the columns 32 w .. of layer 4 in
// FP32 accumulators (176 registers) until the block's last step; the blocks'
// sums are added by reduceAdamKernel.
constexpr int kPartFloats = kMlpParams + 32;  // a block's gradients, then its loss
constexpr size_t kGradFloat4 = 3 * 16 * kBlk;  // a block's GELU derivatives

struct TrainLds {
  bf16x8 x0t[4][2][2][64];      // [wavefront][feature tile][K step][lane]
  bf16x8 ht[3][4][4][2][64];    // [layer][wavefront][unit tile][K step][lane]
  bf16x8 dzt[4][4][2][64];      // [wavefront][unit tile][K step][lane]
  float db[4][3][kHid];         // bias gradients by wavefront
  float db4[4][32];
  float loss[4];
};

// The transposed operands of one 32-unit tile held as K steps a0, a1.
__device__ __forceinline__ f32x16 transposeTile(bf16x8 a0, bf16x8 a1, const bf16x8* ident) {
  f32x16 c = {};
  c = mfma(a0, ident[0], c);
  return mfma(a1, ident[1], c);
}
__device__ __forceinline__ void putOperands(MFCL_LDS bf16x8* o, const f32x16& c, int lane) {
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    bf16x8 v;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = static_cast<__bf16>(c[8 * s + i]);
    o[64 * s + lane] = v;
  }
}

// GELU's derivatives of a layer, 64 per lane in FP32, in the block's stretch
// of the workspace (196 KB a block, which stays in its XCD's L2), 16 bytes per
// lane and step.  In registers beside the gradients' accumulators they spilled
// (2 KB a lane: 233 us a step's kernel; layer 3 alone in registers 167 us; none, as here, 134 us).
struct GradMem {
  float4* p;  // this thread's first entry
  __device__ __forceinline__ void put(int t, const float* g) const {
#pragma unroll
    for (int q = 0; q < 4; ++q) p[(4 * t + q) * kBlk] = make_float4(g[4 * q], g[4 * q + 1], g[4 * q + 2], g[4 * q + 3]);
  }
  __device__ __forceinline__ void get(int t, float* g) const {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 v = p[(4 * t + q) * kBlk];
      g[4 * q] = v.x;
      g[4 * q + 1] = v.y;
      g[4 * q + 2] = v.z;
      g[4 * q + 3] = v.w;
    }
  }
};
// A hidden layer with GELU's derivative: activations to out, their
// transposes to LDS.
template <int KS>
__device__ __forceinline__ void trainDense(const bf16x8* W, const bf16x8* x, const float* bias, int lane, bf16x8* out,
                                           const GradMem& grad, const bf16x8* ident, MFCL_LDS bf16x8* ht) {
  const int h = lane >> 5;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    f32x16 acc = biasTile(bias, t, h);
#pragma unroll
    for (int j = 0; j < KS; ++j) acc = mfma(W[(t * KS + j) * 64 + lane], x[j], acc);
    float g[16];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bf16x8 o;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float z = acc[8 * s + i], q = normalTail(z);
        o[i] = static_cast<__bf16>(geluF(z, q));
        g[8 * s + i] = geluGradF(z, q);
      }
      out[2 * t + s] = o;
    }
    grad.put(t, g);
    putOperands(ht + 128 * t, transposeTile(out[2 * t], out[2 * t + 1], ident), lane);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// dZ of the layer below: dz_out = (W^T dz) * gelu'.
template <int KS>
__device__ __forceinline__ void trainBack(const bf16x8* WT, const bf16x8* dz, const GradMem& grad, int lane, bf16x8* out) {
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    float g[16];
    grad.get(t, g);
    f32x16 acc = {};
#pragma unroll
    for (int j = 0; j < KS; ++j) acc = mfma(WT[(t * KS + j) * 64 + lane], dz[j], acc);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bf16x8 o;
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = static_cast<__bf16>(acc[8 * s + i] * g[8 * s + i]);
      out[2 * t + s] = o;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}
// dZ's transposed operands to LDS and its row sums to the bias gradients.
__device__ __forceinline__ void putDz(const bf16x8* dz, const bf16x8* ident, MFCL_LDS bf16x8* dzt, int lane, float* db) {
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const f32x16 c = transposeTile(dz[2 * t], dz[2 * t + 1], ident);
    putOperands(dzt + 128 * t, c, lane);
    float s = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) s += c[r];
    db[t] += s;
    __builtin_amdgcn_sched_barrier(0);
  }
}
// acc[n] += dZ tile (all four wavefronts' rows) . H tile n
template <int NT>
__device__ __forceinline__ void weightGrad(const MFCL_LDS bf16x8* dzt, int mt, const MFCL_LDS bf16x8* ht, int wave_stride,
                                           f32x16* acc, int lane) {
#pragma unroll
  for (int w = 0; w < 4; ++w)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const bf16x8 a = dzt[((w * 4 + mt) * 2 + s) * 64 + lane];
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = mfma(a, ht[w * wave_stride + (t * 2 + s) * 64 + lane], acc[t]);
    }
}
template <int NT>
__device__ __forceinline__ void storeGrad(float* W, int ld, int m0, int n0, const f32x16* acc, int lane) {
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      W[(m0 + 8 * (r / 4) + 4 * (lane >> 5) + (r % 4)) * ld + n0 + 32 * t + (lane & 31)] = acc[t][r];
}

__global__ void __launch_bounds__(kBlk, 1) mlpTrainFused(const float* xf, const float* target, uint64_t n,
                                                         const bf16x8* pack, const float* bias, float inv_count,
                                                         float wd, float* part, float4* gelu_grad) {
  extern __shared__ __align__(16) char lds_raw[];
  MFCL_LDS TrainLds* L = (MFCL_LDS TrainLds*)((MFCL_LDS char*)(lds_raw));
  const int lane = threadIdx.x & 63, h = lane >> 5, wv = threadIdx.x >> 6;
  // identity operands for activations (units in the accumulators' order) and
  // for features (natural order)
  bf16x8 ident[2], ident0[2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      ident[s][i] = static_cast<__bf16>((lane & 31) == 16 * s + 8 * (i / 4) + 4 * h + (i % 4) ? 1.f : 0.f);
      ident0[s][i] = static_cast<__bf16>((lane & 31) == 16 * s + 8 * h + i ? 1.f : 0.f);
    }
  f32x16 gw1[2] = {}, gw2[4] = {}, gw3[4] = {}, gw4[1] = {};
  float db1[4] = {0, 0, 0, 0}, db2[4] = {0, 0, 0, 0}, db3[4] = {0, 0, 0, 0}, db4 = 0.f, loss = 0.f;
  const GradMem g1{gelu_grad + blockIdx.x * kGradFloat4 + threadIdx.x};
  const GradMem g2{g1.p + 16 * kBlk}, g3{g2.p + 16 * kBlk};
  MFCL_LDS bf16x8* dzt = &L->dzt[wv][0][0][0];
  const MFCL_LDS bf16x8* dz_all = &L->dzt[0][0][0][0];
  for (uint64_t base = static_cast<uint64_t>(blockIdx.x) * 128; base < n; base += static_cast<uint64_t>(gridDim.x) * 128) {
    // opaque, so that the weights and biases are read again for each step:
    // hoisted out of the loop they would fill the registers several times over
    asm volatile("" : "+s"(pack), "+s"(bias));
    const bf16x8* W1 = pack;
    const bf16x8* W2 = W1 + kPackL1 * 64;
    const bf16x8* W3 = W2 + kPackL2 * 64;
    const bf16x8* W4 = W3 + kPackL3 * 64;
    const bf16x8* T4 = W4 + kPackL4 * 64;
    const bf16x8* T3 = T4 + kPackT4 * 64;
    const bf16x8* T2 = T3 + kPackT3 * 64;
    const uint64_t i = base + 32 * wv + (lane & 31);
    bf16x8 a[8], b[8];
    {
      bf16x8 x0[4];
      featureOperands(xf, i, n, h, x0);
#pragma unroll
      for (int t = 0; t < 2; ++t)
        putOperands(&L->x0t[wv][t][0][0], transposeTile(x0[2 * t], x0[2 * t + 1], ident0), lane);
      trainDense<4>(W1, x0, bias, lane, a, g1, ident, &L->ht[0][wv][0][0][0]);
    }
    trainDense<8>(W2, a, bias + kHid, lane, b, g2, ident, &L->ht[1][wv][0][0][0]);
    trainDense<8>(W3, b, bias + 2 * kHid, lane, a, g3, ident, &L->ht[2][wv][0][0][0]);
    // outputs and loss: mean over valid rows of (1 - cos(y[0:3], t[0:3])) +
    // wd (y3 - t3)^2; rows with a zero target direction are masked.  Row
    // lane % 32 is in the lanes below 32.
    f32x16 y = {};
#pragma unroll
    for (int j = 0; j < 8; ++j) y = mfma(W4[j * 64 + lane], a[j], y);
    bf16x8 dy[2] = {};
    if (h == 0 && i < n) {
      const float* t = target + 4 * i;
      const float* b4 = bias + 3 * kHid;
      const float y0 = y[0] + b4[0], y1 = y[1] + b4[1], y2 = y[2] + b4[2], y3 = y[3] + b4[3];
      const float tn = sqrtf(t[0] * t[0] + t[1] * t[1] + t[2] * t[2]);
      if (tn > 0.f) {
        const float yn = fmaxf(sqrtf(y0 * y0 + y1 * y1 + y2 * y2), 1e-12f);
        const float c = (y0 * t[0] + y1 * t[1] + y2 * t[2]) / (yn * tn);
        const float e = y3 - t[3];
        loss += (1.f - c + wd * e * e) * inv_count;
        dy[0][0] = static_cast<__bf16>(-(t[0] / tn - c * y0 / yn) / yn * inv_count);
        dy[0][1] = static_cast<__bf16>(-(t[1] / tn - c * y1 / yn) / yn * inv_count);
        dy[0][2] = static_cast<__bf16>(-(t[2] / tn - c * y2 / yn) / yn * inv_count);
        dy[0][3] = static_cast<__bf16>(2.f * wd * e * inv_count);
      }
    }
    // layer 4
    {
      const f32x16 c = transposeTile(dy[0], dy[1], ident);
      putOperands(dzt, c, lane);
#pragma unroll
      for (int r = 0; r < 16; ++r) db4 += c[r];
    }
    trainBack<1>(T4, dy, g3, lane, b);
    __syncthreads();
    weightGrad<1>(dz_all, 0, &L->ht[2][0][wv][0][0], 512, gw4, lane);
    __syncthreads();
    // layer 3
    putDz(b, ident, dzt, lane, db3);
    trainBack<8>(T3, b, g2, lane, a);
    __syncthreads();
    weightGrad<4>(dz_all, wv, &L->ht[1][0][0][0][0], 512, gw3, lane);
    __syncthreads();
    // layer 2
    putDz(a, ident, dzt, lane, db2);
    trainBack<8>(T2, a, g1, lane, b);
    __syncthreads();
    weightGrad<4>(dz_all, wv, &L->ht[0][0][0][0][0], 512, gw2, lane);
    __syncthreads();
    // layer 1
    putDz(b, ident, dzt, lane, db1);
    __syncthreads();
    weightGrad<2>(dz_all, wv, &L->x0t[0][0][0][0], 256, gw1, lane);
    __syncthreads();
  }
  float* P = part + static_cast<size_t>(blockIdx.x) * kPartFloats;
  storeGrad<2>(P + kOffW1, kMlpInPad, 32 * wv, 0, gw1, lane);
  storeGrad<4>(P + kOffW2, kHid, 32 * wv, 0, gw2, lane);
  storeGrad<4>(P + kOffW3, kHid, 32 * wv, 0, gw3, lane);
  storeGrad<1>(P + kOffW4, kHid, 0, 32 * wv, gw4, lane);
  // bias gradients and loss: lanes l and l + 32 hold the same unit's halves
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const float s1 = db1[t] + __shfl_xor(db1[t], 32), s2 = db2[t] + __shfl_xor(db2[t], 32),
                s3 = db3[t] + __shfl_xor(db3[t], 32);
    if (h == 0) {
      L->db[wv][0][32 * t + lane] = s1;
      L->db[wv][1][32 * t + lane] = s2;
      L->db[wv][2][32 * t + lane] = s3;
    }
  }
  const float s4 = db4 + __shfl_xor(db4, 32);
  if (h == 0) L->db4[wv][lane] = s4;
  for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off);
  if (lane == 0) L->loss[wv] = loss;
  __syncthreads();
  auto sum4 = [](const MFCL_LDS float* p, int stride) { return (p[0] + p[stride]) + (p[2 * stride] + p[3 * stride]); };
  for (int k = threadIdx.x; k < 3 * kHid; k += kBlk) {
    const int off = k < kHid ? kOffB1 : (k < 2 * kHid ? kOffB2 : kOffB3);
    P[off + k % kHid] = sum4(&L->db[0][0][0] + k, 3 * kHid);
  }
  if (threadIdx.x < 32) {
    P[kOffB4 + threadIdx.x] = sum4(&L->db4[0][0] + threadIdx.x, 32);
    P[kMlpParams + threadIdx.x] = threadIdx.x == 0 ? sum4(&L->loss[0], 1) : 0.f;
  }
}

// Sums the blocks' partial gradients (and losses), 64 parameters per block
// of 256 threads, each parameter's partials split over four of them and
// added in a fixed order; then Adam on the FP32 master parameters.  Padding
// entries have zero gradients and stay zero.
struct AdamArgs {
  float* p;
  float* m;
  float* v;
  float lr, b1, b2, eps, c1, c2;
  int apply;
};
__global__ void __launch_bounds__(kBlk) reduceAdamKernel(const float* part, int n_part, float* grad, float* loss,
                                                         AdamArgs a) {
  __shared__ float red[4][64];
  const int g = threadIdx.x >> 6, k = threadIdx.x & 63;
  const int i = blockIdx.x * 64 + k;
  float s = 0.f;
  if (i < kPartFloats)
#pragma unroll 8
    for (int b = g; b < n_part; b += 4) s += part[static_cast<size_t>(b) * kPartFloats + i];
  red[g][k] = s;
  __syncthreads();
  if (g != 0 || i >= kPartFloats) return;
  s = (red[0][k] + red[1][k]) + (red[2][k] + red[3][k]);
  if (i >= kMlpParams) {
    if (i == kMlpParams) *loss = s;
    return;
  }
  grad[i] = s;
  if (!a.apply) return;
  const float mi = a.b1 * a.m[i] + (1.f - a.b1) * s;
  const float vi = a.b2 * a.v[i] + (1.f - a.b2) * s * s;
  a.m[i] = mi;
  a.v[i] = vi;
  a.p[i] -= a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
}

// ------------------------------------------------------------- host side
namespace {

int ensureMlp(mfcl_ctx* ctx) {
  if (ctx->mlp.params) return MFCL_OK;
  ctx->err = "MLP parameters not initialised (mfcl_mlp_init or mfcl_mlp_set_params)";
  return MFCL_E_STATE;
}

const uint4* packOf(const mfcl_ctx* ctx) { return static_cast<const uint4*>(ctx->mlp.pack); }
const float* packBias(const mfcl_ctx* ctx) {
  return reinterpret_cast<const float*>(static_cast<const char*>(ctx->mlp.pack) + kPackBytes);
}

// Refreshes the BF16 weight images from the FP32 master parameters.
void castWeights(mfcl_ctx* ctx, hipStream_t s) {
  auto& M = ctx->mlp;
  const int T = 256;
  packKernel<<<(kPackBlocks * 64 * 8 + T - 1) / T, T, 0, s>>>(M.params, reinterpret_cast<__bf16*>(M.pack),
                                                               const_cast<float*>(packBias(ctx)));
}

// Blocks of a training step: one per CU, at most one per 128 rows.
unsigned trainBlocks(const mfcl_ctx* ctx, uint64_t rows) {
  return static_cast<unsigned>(std::min<uint64_t>((rows + 127) / 128, static_cast<uint64_t>(ctx->n_cu)));
}

// Workspace of a block: its partial gradients and GELU derivatives.
constexpr size_t kBlockBytes = sizeof(float) * kPartFloats + sizeof(float4) * kGradFloat4;

int checkRows(mfcl_ctx* ctx, uint64_t rows) {
  if (rows <= ctx->mlp.ws_rows) return MFCL_OK;
  ctx->err = "MLP workspace too small for " + std::to_string(rows) +
             " rows: call mfcl_reserve(ctx, MFCL_WS_MLP, rows) first";
  return MFCL_E_STATE;
}

}  // namespace

int mlpReserve(mfcl_ctx* ctx, uint64_t rows) {
  if (rows > (1ull << 26)) {
    ctx->err = "MLP rows out of range (<= 2^26)";
    return MFCL_E_INVALID;
  }
  if (rows <= ctx->mlp.ws_rows && ctx->mlp.ws.p) return MFCL_OK;
  const uint64_t most = std::max<uint64_t>(ctx->mlp.ws_rows, rows + rows / 4 + 32);
  if (int rc = ensure(ctx, ctx->mlp.ws, kBlockBytes * trainBlocks(ctx, most))) return rc;
  ctx->mlp.ws_rows = most;
  return MFCL_OK;
}

int mlpInit(mfcl_ctx* ctx, uint64_t seed) {
  std::vector<float> p(kMlpParams, 0.f);
  std::mt19937_64 rng(seed);
  auto fill = [&](int off, int rows, int cols, int fan_in, int fan_out, int valid_rows, int valid_cols) {
    const double a = std::sqrt(6.0 / (fan_in + fan_out));
    std::uniform_real_distribution<double> U(-a, a);
    for (int r = 0; r < rows; ++r)
      for (int c = 0; c < cols; ++c)
        p[off + r * cols + c] = (r < valid_rows && c < valid_cols) ? static_cast<float>(U(rng)) : 0.f;
  };
  fill(kOffW1, kHid, kMlpInPad, kMlpIn, kHid, kHid, kMlpIn);
  fill(kOffW2, kHid, kHid, kHid, kHid, kHid, kHid);
  fill(kOffW3, kHid, kHid, kHid, kHid, kHid, kHid);
  fill(kOffW4, kMlpOutPad, kHid, kHid, kMlpOut, kMlpOut, kHid);
  return mlpSetParams(ctx, p.data(), kMlpParams, true);
}

int mlpSetParams(mfcl_ctx* ctx, const float* host, int n, bool reset_opt) {
  if (n != kMlpParams) {
    ctx->err = "expected " + std::to_string(kMlpParams) + " parameters";
    return MFCL_E_INVALID;
  }
  auto& M = ctx->mlp;
  if (!M.params) {
    const size_t fb = static_cast<size_t>(kMlpParams) * 4;
    MFCL_HIP_TRY(ctx, hipMalloc(&M.params, fb));
    MFCL_HIP_TRY(ctx, hipMalloc(&M.grad, fb));
    MFCL_HIP_TRY(ctx, hipMalloc(&M.m, fb));
    MFCL_HIP_TRY(ctx, hipMalloc(&M.v, fb));
    MFCL_HIP_TRY(ctx, hipMalloc(&M.loss, 256));
    MFCL_HIP_TRY(ctx, hipMalloc(&M.pack, kPackBytes + kPackBiasFloats * 4));
  }
  MFCL_HIP_TRY(ctx, hipMemcpyAsync(M.params, host, static_cast<size_t>(kMlpParams) * 4, hipMemcpyHostToDevice,
                                   ctx->stream));
  if (reset_opt) {
    fillKernel<<<(kMlpParams + 255) / 256, 256, 0, ctx->stream>>>(M.m, kMlpParams, 0.f);
    fillKernel<<<(kMlpParams + 255) / 256, 256, 0, ctx->stream>>>(M.v, kMlpParams, 0.f);
    M.step = 0;
  }
  castWeights(ctx, ctx->stream);
  MFCL_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
  return MFCL_OK;
}

int mlpGetParams(mfcl_ctx* ctx, float* host, int n, float* grad_host) {
  if (int rc = ensureMlp(ctx)) return rc;
  if (n != kMlpParams) {
    ctx->err = "expected " + std::to_string(kMlpParams) + " parameters";
    return MFCL_E_INVALID;
  }
  MFCL_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
  if (host) MFCL_HIP_TRY(ctx, hipMemcpy(host, ctx->mlp.params, static_cast<size_t>(n) * 4, hipMemcpyDeviceToHost));
  if (grad_host)
    MFCL_HIP_TRY(ctx, hipMemcpy(grad_host, ctx->mlp.grad, static_cast<size_t>(n) * 4, hipMemcpyDeviceToHost));
  return MFCL_OK;
}

int mlpFeatures(mfcl_ctx* ctx, const uint32_t* pa, const uint32_t* pb, const float* posea, const float* poseb,
                uint64_t n, float* xf_out, hipStream_t s) {
  if (!ctx->d_desc) {
    ctx->err = "no shapes uploaded";
    return MFCL_E_STATE;
  }
  if (n == 0) return MFCL_OK;
  featureKernel<<<static_cast<unsigned>((n + kBlk - 1) / kBlk), kBlk, 0, s>>>(
      pa, pb, posea, poseb, ctx->d_desc, ctx->n_shapes, n, xf_out);
  MFCL_HIP_TRY(ctx, hipGetLastError());
  return MFCL_OK;
}

int mlpGuess(mfcl_ctx* ctx, const uint32_t* pa, const uint32_t* pb, const float* posea, const float* poseb,
             uint64_t n, float* guess3, float* dist, hipStream_t s) {
  if (int rc = ensureMlp(ctx)) return rc;
  if (!ctx->d_desc) {
    ctx->err = "no shapes uploaded";
    return MFCL_E_STATE;
  }
  if (n == 0) return MFCL_OK;
  if (ctx->timing) MFCL_HIP_TRY(ctx, hipEventRecord(ctx->ev[8], s));
  const size_t lds = kPackFwdBytes + kPackBiasFloats * 4;
  const uint64_t ntiles = (n + 31) / 32;
  // wavefronts per block: more of them share a copy of the weights and hide
  // each other's waits, once there is a tile for each (1,048,576 pairs: 332,
  // 230, 205 us with 4, 8, 16; 4,000 pairs: 14, 17, 27 us)
  const uint64_t cus = static_cast<uint64_t>(ctx->n_cu);
  const int by_size = ntiles >= 16 * cus ? 16 : (ntiles >= 8 * cus ? 8 : 4);
  const int waves = ctx->tune.mlp_waves ? ctx->tune.mlp_waves : by_size;
  // persistent: at most one block per CU (the weights fill most of its LDS)
  const uint64_t want = (ntiles + waves - 1) / waves;
  const uint64_t cap = static_cast<uint64_t>(ctx->n_cu);
  const unsigned grid = static_cast<unsigned>(want < cap ? want : cap);
  const uint4* pk = packOf(ctx);
  const float* pb4 = packBias(ctx);
  const int pol = ctx->tune.guess_policy;
  if (waves == 16)
    mlpGuessFused<1024><<<grid, 1024, lds, s>>>(pa, pb, posea, poseb, ctx->d_desc, ctx->n_shapes, n, pk, pb4, pol,
                                                guess3, dist);
  else if (waves == 8)
    mlpGuessFused<512><<<grid, 512, lds, s>>>(pa, pb, posea, poseb, ctx->d_desc, ctx->n_shapes, n, pk, pb4, pol,
                                              guess3, dist);
  else
    mlpGuessFused<256><<<grid, 256, lds, s>>>(pa, pb, posea, poseb, ctx->d_desc, ctx->n_shapes, n, pk, pb4, pol,
                                              guess3, dist);
  if (ctx->timing) MFCL_HIP_TRY(ctx, hipEventRecord(ctx->ev[9], s));
  MFCL_HIP_TRY(ctx, hipGetLastError());
  return MFCL_OK;
}

int mlpForwardFeat(mfcl_ctx* ctx, const float* xf, uint64_t n, float* y4_out, hipStream_t s) {
  if (int rc = ensureMlp(ctx)) return rc;
  if (n == 0) return MFCL_OK;
  const uint64_t want = (n + 255) / 256;  // 8 wavefronts of 32 rows
  const unsigned grid = static_cast<unsigned>(std::min<uint64_t>(want, static_cast<uint64_t>(ctx->n_cu)));
  mlpForwardFused<<<grid, 512, kPackFwdBytes + kPackBiasFloats * 4, s>>>(xf, n, packOf(ctx), packBias(ctx), y4_out);
  MFCL_HIP_TRY(ctx, hipGetLastError());
  return MFCL_OK;
}

int mlpTrainStep(mfcl_ctx* ctx, const float* xf, const float* target4, uint64_t n, const float* hyper,
                 int apply_update, float* loss_out, hipStream_t s) {
  if (int rc = ensureMlp(ctx)) return rc;
  if (n == 0 || n > (1ull << 26)) {
    ctx->err = "training batch size out of range (1 .. 2^26)";
    return MFCL_E_INVALID;
  }
  if (int rc = checkRows(ctx, n)) return rc;
  auto& M = ctx->mlp;
  const unsigned nb = trainBlocks(ctx, n);
  float4* gelu_grad = static_cast<float4*>(M.ws.p);
  float* part = reinterpret_cast<float*>(gelu_grad + nb * kGradFloat4);
  const float wd = hyper ? hyper[5] : 1.0f;
  mlpTrainFused<<<nb, kBlk, sizeof(TrainLds), s>>>(xf, target4, n, reinterpret_cast<const bf16x8*>(packOf(ctx)),
                                                   packBias(ctx), 1.0f / static_cast<float>(n), wd, part, gelu_grad);
  AdamArgs a{M.params, M.m, M.v, 0, 0, 0, 0, 1, 1, apply_update != 0 ? 1 : 0};
  if (apply_update) {
    a.lr = hyper ? hyper[0] : 1e-3f;
    a.b1 = hyper ? hyper[1] : 0.9f;
    a.b2 = hyper ? hyper[2] : 0.999f;
    a.eps = hyper ? hyper[3] : 1e-8f;
    M.step += 1;
    a.c1 = 1.f - std::pow(a.b1, static_cast<float>(M.step));
    a.c2 = 1.f - std::pow(a.b2, static_cast<float>(M.step));
  }
  reduceAdamKernel<<<(kPartFloats + 63) / 64, kBlk, 0, s>>>(part, static_cast<int>(nb), M.grad, M.loss, a);
  if (apply_update) castWeights(ctx, s);
  if (loss_out) MFCL_HIP_TRY(ctx, hipMemcpyAsync(loss_out, M.loss, 4, hipMemcpyDeviceToHost, s));
  MFCL_HIP_TRY(ctx, hipGetLastError());
  return MFCL_OK;
}

void mlpFree(mfcl_ctx* ctx) {
  auto& M = ctx->mlp;
  for (void* p : {static_cast<void*>(M.params), static_cast<void*>(M.grad), static_cast<void*>(M.m),
                  static_cast<void*>(M.v), static_cast<void*>(M.loss), M.ws.p, M.pack})
    if (p) (void)hipFree(p);
  M = MlpState{};
}

}  // namespace mfcl
