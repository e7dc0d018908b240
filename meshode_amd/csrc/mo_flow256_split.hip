// The 3-256-256-256-3 softplus field's RK4 step and its adjoint with the
// 256 x 256 products on bf16 MFMA at 32-bit accuracy.
//
// An FP32 number is the exact sum of three bf16 (high, middle, low: 3 x 8
// significant bits) if it is below 3.39e38, bf16's largest, and large enough
// for its low part to be a normal bf16 (the matrix cores drop the bits of
// others): from 2^-110 on, which the factors along a gradient's way turn into
// about 2^-100 for dL/dy1 (2^-110 there gives 6e-6, 2^-115 2e-4).  A product
// of two such sums is formed from the six partial products of order 2^-16 and
// above (hh, hm, mh, mm, hl, lh); the three left out are below 2^-25 of the
// product, under the rounding of an FP32 product, and the sums are
// accumulated in FP32 as before; against FP64 the results are as near as with
// FP32 MFMA or nearer (parameter gradients of 4000 points over 3 steps 1.8e-7
// at most, there 3.4e-7).  Six bf16 products cost 6/16 of the one
// FP32 product they replace (v_mfma_f32_32x32x16_bf16 does 1024 flops a cycle
// on a SIMD, v_mfma_f32_32x32x2_f32 64), so the bound rises from 157 to
// 417 TFLOP/s of FP32 work.  The bf16 MFMA drops the bits of an
// addend below its sum's range downwards, a bias that a sum over 10^5 points
// of random sign shows (parameter gradients off by 5e-6); odd points
// therefore run through the products negated, and odd workgroups of the
// weight-gradient product form -dW, which cancels it.  (A non-finite
// activation gives NaN: its middle and low parts are NaN.)
//
// Forward (k_flow256_fwd): a workgroup of 8 wavefronts takes 64 points
// through all four stages.  The activations of the 64 points are three bf16
// planes in LDS, [plane][k / 8][point][8] (96 KiB, one buffer: a layer's
// outputs wait in registers, already split, until every wave has read its
// inputs): the B operand of the MFMA is one conflict-free 16-byte read, and
// with the weights as A operand (M = units) a lane ends up with four
// consecutive units of one point, one 8-byte store per plane.  Wave w
// computes units [32 w, 32 w + 32) for both 32-point blocks, so each weight
// fragment, streamed from L2 (393 KB a layer), serves 12 MFMAs.  The five
// small products are summed apart from the large one: the long sum is then
// rounded 16 times and not 96, which halves the errors.  The 3 -> 256 and
// 256 -> 3 layers are on the VALU, the latter straight from the accumulators.
//
// Adjoint (k_flow256_adj, k_flow256_adj_dw): the forward keeps the stage
// inputs (48 B a point and step).  Per stage, last first, the backward
// recomputes the three hidden layers, keeping softplus'(A2) in the registers
// of the lane that will need it, and walks back through the transposed
// products; H1, H2, dA2 and dA3 go to memory transposed ([unit][stage point],
// 128-byte rows of 32 points) for the weight-gradient product over the step's
// 4 n stage points, and dW0, db0, dW3, db3 are summed on the spot.  The products' partials are kept per
// workgroup across the steps of an integration and added in FP64 once.
//
// Measured, 55000 points, 16 steps: forward and gradients 54.1 -> 27.0 ms
// with the FP32 MFMA kernels before (whose adjoint also moved 3.8 GB a step
// through memory, now 1.8 GB); a forward step 676 -> 356 us (983 TFLOP/s of
// bf16 products, where an 8192^3 library product reaches 1118), an adjoint
// step 967 + 390 us (k_flow256_adj spills 33 VGPRs, 132 bytes a lane, and
// k_flow256_adj_dw 6); 5001 points forward 2980 -> 870 us for 16 steps, on 157
// workgroups of 32 points (99 CUs have none).  MFMA busy 46, 32 and 37% of the
// time (forward, adjoint, weight gradients).
#include <algorithm>

#include "mo_common.h"
#include "mo_flow256.h"

#define MO_EXPORT extern "C" __attribute__((visibility("default")))

namespace mo {
namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));

constexpr int kPts = 64;
constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int kPlaneW = kSplitPlane / 4;     // 16-byte words of a weight plane (8192)
// weight steps in registers: the adjoint has no room for four (27.4 against
// 27.0 ms a training step)
constexpr int kRingFwd = 4, kRingAdj = 2;
constexpr int kXPlane = 32 * kPts;           // 16-byte words of an activation plane

// field constants in LDS: W0's columns, b0, b1, b2, W3's rows
enum { cW0 = 0, cB0 = 3 * kH, cB1 = 4 * kH, cB2 = 5 * kH, cW3 = 6 * kH, cNum = 9 * kH };

__device__ __forceinline__ float softplus(float x) {
  const float e = __builtin_amdgcn_exp2f(-fabsf(x) * 1.4426950408889634f);
  return fmaxf(x, 0.f) + __builtin_amdgcn_logf(1.f + e) * 0.6931471805599453f;
}

// softplus and its derivative 1 / (1 + exp(-x)) from the one exponential
__device__ __forceinline__ float softplus_d(float x, float& d) {
  const float e = __builtin_amdgcn_exp2f(-fabsf(x) * 1.4426950408889634f);
  const float r = __builtin_amdgcn_rcpf(1.f + e);
  d = x >= 0.f ? r : e * r;
  return fmaxf(x, 0.f) + __builtin_amdgcn_logf(1.f + e) * 0.6931471805599453f;
}

__device__ __forceinline__ float flip(float v, unsigned sign) { return __uint_as_float(__float_as_uint(v) ^ sign); }

// four values, negated where `sign` is the sign bit, -> their three bf16
// planes (8 bytes each)
__device__ __forceinline__ void split4(const float (&v)[4], unsigned sign, uint2 (&o)[3]) {
  float r[4] = {flip(v[0], sign), flip(v[1], sign), flip(v[2], sign), flip(v[3], sign)};
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    const unsigned lo = __builtin_bit_cast(unsigned, __builtin_convertvector((f2{r[0], r[1]}), b2));
    const unsigned hi = __builtin_bit_cast(unsigned, __builtin_convertvector((f2{r[2], r[3]}), b2));
    o[p] = make_uint2(lo, hi);
    if (p < 2) {
      r[0] -= __uint_as_float(lo << 16);
      r[1] -= __uint_as_float(lo & 0xFFFF0000u);
      r[2] -= __uint_as_float(hi << 16);
      r[3] -= __uint_as_float(hi & 0xFFFF0000u);
    }
  }
}

// planes of units [32 w + 8 g + 4 (l / 32), + 4) of point p
__device__ __forceinline__ void store_planes(uint4* X, int w, int g, int hi, int p, const uint2 (&o)[3]) {
#pragma unroll
  for (int pl = 0; pl < 3; ++pl) reinterpret_cast<uint2*>(X + pl * kXPlane + (4 * w + g) * kPts + p)[hi] = o[pl];
}

// acc[q] += W X for this wave's 32 units and the point blocks q < NB: 16
// steps of k = 16, six products each, the small ones first.
// kR - 1 steps' weights are in flight.
template <int NB, int kR>
__device__ __forceinline__ void gemm(const float* __restrict__ Wf, const uint4* X, int w, int l, v16f (&acc)[2]) {
  const uint4* __restrict__ A = reinterpret_cast<const uint4*>(Wf) + w * (16 * 64) + l;
  const uint4* B = X + (l >> 5) * kPts + (l & 31);
  v16f low[2] = {v16f{0}, v16f{0}};
  uint4 a[kR][3];
#pragma unroll
  for (int d = 0; d < kR - 1; ++d)
#pragma unroll
    for (int p = 0; p < 3; ++p) a[d][p] = A[p * kPlaneW + d * 64];
#pragma unroll kR
  for (int ks = 0; ks < 16; ++ks) {
    const int cur = ks % kR;
    if (ks + kR - 1 < 16) {
#pragma unroll
      for (int p = 0; p < 3; ++p) a[(ks + kR - 1) % kR][p] = A[p * kPlaneW + (ks + kR - 1) * 64];
    }
    b8 bx[NB][3];
#pragma unroll
    for (int q = 0; q < NB; ++q)
#pragma unroll
      for (int p = 0; p < 3; ++p) bx[q][p] = __builtin_bit_cast(b8, B[p * kXPlane + 2 * ks * kPts + 32 * q]);
    constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        v16f& d = t < 5 ? low[q] : acc[q];
        d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8, a[cur][pa[t]]), bx[q][pb[t]], d, 0, 0, 0);
      }
  }
#pragma unroll
  for (int q = 0; q < NB; ++q) acc[q] += low[q];
}

__device__ __forceinline__ void load_constants(float* Wc, const float* __restrict__ P) {
  for (int u = threadIdx.x; u < kH; u += kThreads) {
    const float4 r = *reinterpret_cast<const float4*>(P + kPW0 + 4 * u);
    Wc[cW0 + u] = r.x;
    Wc[cW0 + kH + u] = r.y;
    Wc[cW0 + 2 * kH + u] = r.z;
    Wc[cB0 + u] = P[kPB0 + u];
    Wc[cB1 + u] = P[kPB1 + u];
    Wc[cB2 + u] = P[kPB2 + u];
    for (int c = 0; c < 3; ++c) Wc[cW3 + c * kH + u] = P[kPW3 + c * kH + u];
  }
}

__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }

// the accumulators' start: the layer's bias (units 32 w + 8 g + 4 hi + j)
template <int NB>
__device__ __forceinline__ void set_bias(const float* b, int w, int hi, unsigned sign, v16f (&acc)[2]) {
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const float4 v = ld4(b + 32 * w + 8 * g + 4 * hi);
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      acc[q][4 * g] = flip(v.x, sign);
      acc[q][4 * g + 1] = flip(v.y, sign);
      acc[q][4 * g + 2] = flip(v.z, sign);
      acc[q][4 * g + 3] = flip(v.w, sign);
    }
  }
}

// layer 0 of point x: pre-activations of units 32 w + 8 g + 4 hi + j
__device__ __forceinline__ void layer0(const float* Wc, int u, const float* x, float (&v)[4]) {
  const float4 a = ld4(Wc + cW0 + u), b = ld4(Wc + cW0 + kH + u), c = ld4(Wc + cW0 + 2 * kH + u),
               d = ld4(Wc + cB0 + u);
  v[0] = d.x + a.x * x[0] + b.x * x[1] + c.x * x[2];
  v[1] = d.y + a.y * x[0] + b.y * x[1] + c.y * x[2];
  v[2] = d.z + a.z * x[0] + b.z * x[1] + c.z * x[2];
  v[3] = d.w + a.w * x[0] + b.w * x[1] + c.w * x[2];
}

// velocity at the points' x (LDS Z) into part[w][point][3]
template <int NB>
__device__ __forceinline__ void field(const float* __restrict__ P, const float* Wc, uint4* X, const float (*Z)[3],
                                      float (*part)[kPts][3], int w, int l) {
  const int hi = l >> 5, pl = l & 31;
  const unsigned sign = (unsigned)pl << 31;   // odd points run negated (see the top of the file)
#pragma unroll
  for (int q = 0; q < NB; ++q) {
    const float x[3] = {Z[32 * q + pl][0], Z[32 * q + pl][1], Z[32 * q + pl][2]};
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float v[4];
      layer0(Wc, 32 * w + 8 * g + 4 * hi, x, v);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = softplus(v[j]);
      uint2 o[3];
      split4(v, sign, o);
      store_planes(X, w, g, hi, 32 * q + pl, o);
    }
  }
  __syncthreads();
  v16f acc[2];
  set_bias<NB>(Wc + cB1, w, hi, sign, acc);
  gemm<NB, kRingFwd>(P + kPSplit, X, w, l, acc);
  uint2 o[NB][4][3];
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = softplus(flip(acc[q][4 * g + j], sign));
      split4(v, sign, o[q][g]);
    }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int g = 0; g < 4; ++g) store_planes(X, w, g, hi, 32 * q + pl, o[q][g]);
  __syncthreads();
  set_bias<NB>(Wc + cB2, w, hi, sign, acc);
  gemm<NB, kRingFwd>(P + kPSplit + kSplitLayer, X, w, l, acc);
#pragma unroll
  for (int q = 0; q < NB; ++q) {
    float s0 = 0.f, s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int u = 32 * w + 8 * g + 4 * hi;
      const float4 a = ld4(Wc + cW3 + u), b = ld4(Wc + cW3 + kH + u), c = ld4(Wc + cW3 + 2 * kH + u);
      const float h0 = softplus(flip(acc[q][4 * g], sign)), h1 = softplus(flip(acc[q][4 * g + 1], sign)), h2 = softplus(flip(acc[q][4 * g + 2], sign)),
                  h3 = softplus(flip(acc[q][4 * g + 3], sign));
      s0 += a.x * h0 + a.y * h1 + a.z * h2 + a.w * h3;
      s1 += b.x * h0 + b.y * h1 + b.z * h2 + b.w * h3;
      s2 += c.x * h0 + c.y * h1 + c.z * h2 + c.w * h3;
    }
    s0 += __shfl_xor(s0, 32, 64);
    s1 += __shfl_xor(s1, 32, 64);
    s2 += __shfl_xor(s2, 32, 64);
    if (hi == 0) {
      part[w][32 * q + pl][0] = s0;
      part[w][32 * q + pl][1] = s1;
      part[w][32 * q + pl][2] = s2;
    }
  }
}

// Workgroup b of G takes points [n b / G, n (b + 1) / G) in chunks of 64; a
// chunk of at most 32 points skips the second 32-point block.  Zs (or null):
// the stage inputs [4][n][3].
// Bound: bf16 MFMA (with the weight stream from L2 at half its rate), then
// the softplus / splitting VALU work between a layer's barriers.  Raising the
// wave priority of half the waves, to set the two phases against each other,
// changed nothing.
__global__ __launch_bounds__(kThreads, 2) void k_flow256_fwd(const float* __restrict__ y0, int n,
                                                             const float* __restrict__ P, float h,
                                                             float* __restrict__ y1, float* __restrict__ Zs) {
  __shared__ uint4 X[3 * kXPlane];
  __shared__ __align__(16) float Wc[cNum];
  __shared__ float Y[kPts][3], Z[kPts][3], K[4][kPts][3];
  __shared__ float part[kWaves][kPts][3];
  const int tid = threadIdx.x, l = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int p0 = (int)((long long)n * blockIdx.x / gridDim.x);
  const int p1 = (int)((long long)n * (blockIdx.x + 1) / gridDim.x);
  load_constants(Wc, P);
#pragma unroll 1
  for (int base = p0; base < p1; base += kPts) {
    const int nvalid = min(kPts, p1 - base);
    if (tid < kPts)
      for (int c = 0; c < 3; ++c) Y[tid][c] = tid < nvalid ? y0[3 * (size_t)(base + tid) + c] : 0.5f;
#pragma unroll 1
    for (int s = 0; s < 4; ++s) {
      if (tid < kPts)
        for (int c = 0; c < 3; ++c) {
          const float y = Y[tid][c];
          const float z = s == 0 ? y
                        : s == 1 ? y + h * K[0][tid][c] / 3.0f
                        : s == 2 ? y + h * (K[1][tid][c] - K[0][tid][c] / 3.0f)
                                 : y + h * (K[0][tid][c] - K[1][tid][c] + K[2][tid][c]);
          Z[tid][c] = z - 0.5f;
          if (Zs && tid < nvalid) Zs[((size_t)s * n + base + tid) * 3 + c] = z;
        }
      __syncthreads();
      if (nvalid > 32) field<2>(P, Wc, X, Z, part, w, l);
      else field<1>(P, Wc, X, Z, part, w, l);
      __syncthreads();
      if (tid < kPts)
        for (int c = 0; c < 3; ++c) {
          float o = 0.f;
          for (int q = 0; q < kWaves; ++q) o += part[q][tid][c];
          K[s][tid][c] = P[kPB3 + c] + o;
        }
    }
    if (tid < nvalid)
      for (int c = 0; c < 3; ++c)
        y1[3 * (size_t)(base + tid) + c] =
            Y[tid][c] + h * (K[0][tid][c] + 3.0f * (K[1][tid][c] + K[2][tid][c]) + K[3][tid][c]) * 0.125f;
  }
}

// ---------------------------------------------------------------------------
// Adjoint of one step.

// the workgroup's sums: dW0 [256][3], db0 [256], dW3 [3][256], db3 [3]
constexpr int kAdjSmall = 3 * kH + kH + 3 * kH + 3;
// dW [256][256], db [256] of one of the two hidden products
constexpr int kAdjDw = kH * kH + kH;
constexpr int kTileLd = kPts + 1;    // unit-major FP32 tile, padded: column sums read it without bank conflicts
static_assert(kH * kTileLd * 4 <= 3 * kXPlane * 16, "the tile lies over the planes");

struct AdjSums {
  float w0[3], b0, w3[3], g[3];
};

// One stage for NB point blocks.  Xs: the points' x = z - 0.5, G: dL/dk of
// the stage (0 for points beyond the chunk); T: rows of the chunk's first
// stage point in [4][256][ld]; part gets dL/dz per wave.
template <int NB>
__device__ __forceinline__ void adj_stage(const float* __restrict__ P, const float* Wc, uint4* X,
                                          const float (*Xs)[3], const float (*G)[3], float (*part)[kPts][3],
                                          float* __restrict__ T, long long ld, int nvalid, int w, int l, AdjSums& S) {
  const int hi = l >> 5, pl = l & 31;
  const unsigned sign = (unsigned)pl << 31;   // odd points run negated (see the top of the file)
  float* TL = reinterpret_cast<float*>(X);
  const size_t mat = (size_t)kH * ld;
  float s2[NB][16];
  // a lane's place in the transposed rows: a wave-uniform row start (scalar
  // registers) plus one 32-bit offset
  const unsigned at = (unsigned)(4 * hi * ld) + (unsigned)pl;
  auto put = [&](int m, int g, int j, int q, float v) {
    float* r = T + m * mat + (size_t)(32 * w + 8 * g + j) * ld + 32 * q;
    r[at] = v;
  };
  // H1
#pragma unroll
  for (int q = 0; q < NB; ++q) {
    const float x[3] = {Xs[32 * q + pl][0], Xs[32 * q + pl][1], Xs[32 * q + pl][2]};
    const bool ok = 32 * q + pl < nvalid;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float v[4];
      layer0(Wc, 32 * w + 8 * g + 4 * hi, x, v);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = softplus(v[j]);
        if (ok) put(0, g, j, q, v[j]);
      }
      uint2 o[3];
      split4(v, sign, o);
      __builtin_amdgcn_sched_barrier(0);
      store_planes(X, w, g, hi, 32 * q + pl, o);
    }
  }
  __syncthreads();
  v16f acc[2];
  uint2 o[NB][4][3];
  // H2
  set_bias<NB>(Wc + cB1, w, hi, sign, acc);
  gemm<NB, kRingAdj>(P + kPSplit, X, w, l, acc);
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = softplus_d(flip(acc[q][4 * g + j], sign), s2[q][4 * g + j]);
        if (32 * q + pl < nvalid) put(1, g, j, q, v[j]);
      }
      split4(v, sign, o[q][g]);
      __builtin_amdgcn_sched_barrier(0);
    }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int g = 0; g < 4; ++g) store_planes(X, w, g, hi, 32 * q + pl, o[q][g]);
  __syncthreads();
  // H3 (only its sums with G are needed) and dA3 = (W3^T G) softplus'(A3)
  set_bias<NB>(Wc + cB2, w, hi, sign, acc);
  gemm<NB, kRingAdj>(P + kPSplit + kSplitLayer, X, w, l, acc);
  __syncthreads();       // every wave has read the planes the tile now covers
#pragma unroll
  for (int q = 0; q < NB; ++q) {
    const float g0 = G[32 * q + pl][0], g1 = G[32 * q + pl][1], g2 = G[32 * q + pl][2];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int u = 32 * w + 8 * g + 4 * hi;
      const float4 a = ld4(Wc + cW3 + u), b = ld4(Wc + cW3 + kH + u), c = ld4(Wc + cW3 + 2 * kH + u);
      const float dh[4] = {a.x * g0 + b.x * g1 + c.x * g2, a.y * g0 + b.y * g1 + c.y * g2,
                           a.z * g0 + b.z * g1 + c.z * g2, a.w * g0 + b.w * g1 + c.w * g2};
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float s3;
        TL[(u + j) * kTileLd + 32 * q + pl] = softplus_d(flip(acc[q][4 * g + j], sign), s3);
        v[j] = dh[j] * s3;
        if (32 * q + pl < nvalid) put(3, g, j, q, v[j]);
      }
      split4(v, sign, o[q][g]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();
  const int tu = threadIdx.x & (kH - 1), th = threadIdx.x >> 8;   // column sums: unit, half of the points
  {
    // (a stage's sums first: shorter chains of roundings)
    float a[3] = {0.f, 0.f, 0.f}, b[3] = {0.f, 0.f, 0.f};
#pragma unroll 4
    for (int p = 16 * NB * th; p < 16 * NB * (th + 1); ++p) {
      const float t = TL[tu * kTileLd + p];
      for (int c = 0; c < 3; ++c) {
        a[c] += G[p][c] * t;
        b[c] += G[p][c];
      }
    }
    for (int c = 0; c < 3; ++c) {
      S.w3[c] += a[c];
      S.g[c] += b[c];
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int g = 0; g < 4; ++g) store_planes(X, w, g, hi, 32 * q + pl, o[q][g]);
  __syncthreads();
  // dA2 = (dA3 W2) softplus'(A2)
  acc[0] = acc[1] = v16f{0};
  gemm<NB, kRingAdj>(P + kPSplit + 3 * kSplitLayer, X, w, l, acc);
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = flip(acc[q][4 * g + j], sign) * s2[q][4 * g + j];
        if (32 * q + pl < nvalid) put(2, g, j, q, v[j]);
      }
      split4(v, sign, o[q][g]);
      __builtin_amdgcn_sched_barrier(0);
    }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int g = 0; g < 4; ++g) store_planes(X, w, g, hi, 32 * q + pl, o[q][g]);
  __syncthreads();
  // dA1 = (dA2 W1) softplus'(A1), dz = W0^T dA1
  acc[0] = acc[1] = v16f{0};
  gemm<NB, kRingAdj>(P + kPSplit + 2 * kSplitLayer, X, w, l, acc);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NB; ++q) {
    float d0 = 0.f, d1 = 0.f, d2 = 0.f;
    const float x[3] = {Xs[32 * q + pl][0], Xs[32 * q + pl][1], Xs[32 * q + pl][2]};
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int u = 32 * w + 8 * g + 4 * hi;
      const float4 a = ld4(Wc + cW0 + u), b = ld4(Wc + cW0 + kH + u), c = ld4(Wc + cW0 + 2 * kH + u);
      // softplus'(A1) again from the point, cheaper than 32 registers held
      // through the stage
      float v[4];
      layer0(Wc, u, x, v);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float e = __builtin_amdgcn_exp2f(-fabsf(v[j]) * 1.4426950408889634f);
        const float r = __builtin_amdgcn_rcpf(1.f + e);
        v[j] = flip(acc[q][4 * g + j], sign) * (v[j] >= 0.f ? r : e * r);
        TL[(u + j) * kTileLd + 32 * q + pl] = v[j];
      }
      d0 += a.x * v[0] + a.y * v[1] + a.z * v[2] + a.w * v[3];
      d1 += b.x * v[0] + b.y * v[1] + b.z * v[2] + b.w * v[3];
      d2 += c.x * v[0] + c.y * v[1] + c.z * v[2] + c.w * v[3];
      __builtin_amdgcn_sched_barrier(0);
    }
    d0 += __shfl_xor(d0, 32, 64);
    d1 += __shfl_xor(d1, 32, 64);
    d2 += __shfl_xor(d2, 32, 64);
    if (hi == 0) {
      part[w][32 * q + pl][0] = d0;
      part[w][32 * q + pl][1] = d1;
      part[w][32 * q + pl][2] = d2;
    }
  }
  __syncthreads();
  {
    float a[3] = {0.f, 0.f, 0.f}, b = 0.f;
#pragma unroll 4
    for (int p = 16 * NB * th; p < 16 * NB * (th + 1); ++p) {
      const float t = TL[tu * kTileLd + p];
      for (int c = 0; c < 3; ++c) a[c] += Xs[p][c] * t;
      b += t;
    }
    for (int c = 0; c < 3; ++c) S.w0[c] += a[c];
    S.b0 += b;
  }
}

// Zs [4][n][3]: the step's stage inputs; gy1 = dL/dy1 -> gy0 = dL/dy0; T
// [4][256][4 n]: H1, H2, dA2, dA3, transposed, stage after stage; small
// [G][kAdjSmall]: this workgroup's sums, added to what is there unless
// `first`.  RK4 chain: y1 = y + h (k1 + 3 k2 + 3 k3 + k4) / 8, z2 = y + h k1 / 3,
// z3 = y + h (k2 - k1 / 3), z4 = y + h (k1 - k2 + k3).
__global__ __launch_bounds__(kThreads, 2) void k_flow256_adj(int n, const float* __restrict__ P, float h,
                                                             const float* __restrict__ Zs,
                                                             const float* __restrict__ gy1, float* __restrict__ gy0,
                                                             float* __restrict__ T, float* __restrict__ small,
                                                             int first) {
  __shared__ uint4 X[3 * kXPlane];
  __shared__ __align__(16) float Wc[cNum];
  __shared__ float Xs[kPts][3], DK[4][kPts][3], DY[kPts][3];
  __shared__ float part[kWaves][kPts][3];
  const int tid = threadIdx.x, l = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int p0 = (int)((long long)n * blockIdx.x / gridDim.x);
  const int p1 = (int)((long long)n * (blockIdx.x + 1) / gridDim.x);
  const long long ld = 4LL * n;
  const float third = h / 3.0f;
  AdjSums S = {};
  load_constants(Wc, P);
#pragma unroll 1
  for (int base = p0; base < p1; base += kPts) {
    const int nvalid = min(kPts, p1 - base);
    if (tid < kPts)
      for (int c = 0; c < 3; ++c) {
        const float g = tid < nvalid ? gy1[3 * (size_t)(base + tid) + c] : 0.f;
        DY[tid][c] = g;
        const float a = h * g * 0.125f;
        DK[0][tid][c] = a;
        DK[1][tid][c] = 3.0f * a;
        DK[2][tid][c] = 3.0f * a;
        DK[3][tid][c] = a;
      }
#pragma unroll 1
    for (int s = 3; s >= 0; --s) {
      __syncthreads();       // the last stage's sums have been read
      if (tid < kPts)
        for (int c = 0; c < 3; ++c)
          Xs[tid][c] = tid < nvalid ? Zs[((size_t)s * n + base + tid) * 3 + c] - 0.5f : 0.f;
      __syncthreads();
      float* Tc = T + (size_t)s * n + base;
      if (nvalid > 32) adj_stage<2>(P, Wc, X, Xs, DK[s], part, Tc, ld, nvalid, w, l, S);
      else adj_stage<1>(P, Wc, X, Xs, DK[s], part, Tc, ld, nvalid, w, l, S);
      if (tid < kPts && (nvalid > 32 || tid < 32))
        for (int c = 0; c < 3; ++c) {
          float dz = 0.f;
          for (int q = 0; q < kWaves; ++q) dz += part[q][tid][c];
          DY[tid][c] += dz;
          if (s == 3) {          // z4 = y + h (k1 - k2 + k3)
            DK[0][tid][c] += h * dz;
            DK[1][tid][c] -= h * dz;
            DK[2][tid][c] += h * dz;
          } else if (s == 2) {   // z3 = y + h (k2 - k1 / 3)
            DK[1][tid][c] += h * dz;
            DK[0][tid][c] -= third * dz;
          } else if (s == 1) {   // z2 = y + h k1 / 3
            DK[0][tid][c] += third * dz;
          }
        }
    }
    if (tid < nvalid)
      for (int c = 0; c < 3; ++c) gy0[3 * (size_t)(base + tid) + c] = DY[tid][c];
    __syncthreads();
  }
  // the two halves' sums
  float* R = reinterpret_cast<float*>(X);
  const int u = tid & (kH - 1);
  if (tid >= kH) {
    for (int c = 0; c < 3; ++c) {
      R[c * kH + u] = S.w0[c];
      R[(4 + c) * kH + u] = S.w3[c];
      if (u == 0) R[7 * kH + c] = S.g[c];
    }
    R[3 * kH + u] = S.b0;
  }
  __syncthreads();
  if (tid < kH) {
    float* o = small + (size_t)blockIdx.x * kAdjSmall;
    auto put = [&](int e, float v) { o[e] = first ? v : o[e] + v; };
    for (int c = 0; c < 3; ++c) {
      put(3 * u + c, S.w0[c] + R[c * kH + u]);
      put(4 * kH + c * kH + u, S.w3[c] + R[(4 + c) * kH + u]);
      if (u == 0) put(7 * kH + c, S.g[c] + R[7 * kH + c]);
    }
    put(3 * kH + u, S.b0 + R[3 * kH + u]);
  }
}

// dW1 = dA2^T H1 (blockIdx.y = 0) and dW2 = dA3^T H2 with the bias sums of
// dA2, dA3, over stage points in chunks of 32: workgroup b of G takes chunks
// [C b / G, C (b + 1) / G), splits them into LDS planes ([plane][k / 8][unit]
// [8], the k blocks padded apart) with the next chunk in flight to
// registers; wave (w / 2, w % 2) holds a 64 x 128 block of the product.
// Partials [2][G][kAdjDw], added to what is there unless `first`.
constexpr int kDwPts = 32;
constexpr int kDwKb = kH + 4;                 // 16-byte words of a k block
constexpr int kDwPlane = 4 * kDwKb;
__global__ __launch_bounds__(kThreads, 2) void k_flow256_adj_dw(long long rows, const float* __restrict__ T,
                                                                float* __restrict__ partial, int first) {
  __shared__ uint4 SA[3 * kDwPlane];
  __shared__ uint4 SB[3 * kDwPlane];
  const int tid = threadIdx.x, l = tid & 63, hi = l >> 5, pl = l & 31;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float* D = T + (size_t)(2 + blockIdx.y) * kH * rows;
  const float* Hm = T + (size_t)blockIdx.y * kH * rows;
  const long long nch = (rows + kDwPts - 1) / kDwPts;
  const long long c0 = nch * blockIdx.x / gridDim.x, c1 = nch * (blockIdx.x + 1) / gridDim.x;
  const unsigned sign = (blockIdx.x & 1u) << 31;   // odd workgroups form -dW
  const int seg = tid & 7, r8 = tid >> 3;    // four points of rows r8 + 64 i
  v16f acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = v16f{0};
  float db[4] = {0.f, 0.f, 0.f, 0.f};
  float4 pf[8];
  auto fetch = [&](long long c) {
    const long long at = c * kDwPts + 4 * seg;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float* src = i < 4 ? D + (size_t)(r8 + 64 * i) * rows : Hm + (size_t)(r8 + 64 * (i - 4)) * rows;
      pf[i] = at < rows ? *reinterpret_cast<const float4*>(src + at) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  if (c0 < c1) fetch(c0);
#pragma unroll 1
  for (long long c = c0; c < c1; ++c) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float v[4] = {pf[i].x, pf[i].y, pf[i].z, pf[i].w};
      uint2 o[3];
      split4(v, i < 4 ? sign : 0u, o);
      uint4* dst = (i < 4 ? SA : SB) + (seg >> 1) * kDwKb + r8 + 64 * (i & 3);
#pragma unroll
      for (int p = 0; p < 3; ++p) reinterpret_cast<uint2*>(dst + p * kDwPlane)[seg & 1] = o[p];
      if (i < 4) db[i] += (v[0] + v[1]) + (v[2] + v[3]);
    }
    __syncthreads();
    if (c + 1 < c1) fetch(c + 1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int kb = (2 * ks + hi) * kDwKb;
      b8 a[2][3];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int p = 0; p < 3; ++p)
          a[i][p] = __builtin_bit_cast(b8, SA[p * kDwPlane + kb + 64 * (w >> 1) + 32 * i + pl]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        b8 b[3];
#pragma unroll
        for (int p = 0; p < 3; ++p)
          b[p] = __builtin_bit_cast(b8, SB[p * kDwPlane + kb + 128 * (w & 1) + 32 * j + pl]);
        // the small products are summed apart, so that the long sum is
        // rounded twice a step and not six times
        constexpr int pa[5] = {2, 0, 1, 1, 0}, pb[5] = {0, 2, 1, 0, 1};
        v16f low[2] = {v16f{0}, v16f{0}};
#pragma unroll
        for (int t = 0; t < 5; ++t)
#pragma unroll
          for (int i = 0; i < 2; ++i)
            low[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][pa[t]], b[pb[t]], low[i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][0], b[0], acc[i][j], 0, 0, 0);
          acc[i][j] += low[i];
        }
      }
    }
  }
  float* out = partial + ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * kAdjDw;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float* o = out + (64 * (w >> 1) + 32 * i + 8 * (r >> 2) + 4 * hi + (r & 3)) * kH + 128 * (w & 1) + 32 * j + pl;
        const float v = flip(acc[i][j][r], sign);
        *o = first ? v : *o + v;
      }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float v = db[i];
    for (int o = 1; o < 8; o <<= 1) v += __shfl_xor(v, o, 64);
    if (seg == 0) {
      float* o = out + kH * kH + r8 + 64 * i;
      *o = first ? v : *o + v;
    }
  }
}

// the eight parameter gradients from the partials, rows added in order (FP64)
struct AdjOut {
  float *W0, *b0, *W1, *b1, *W2, *b2, *W3, *b3;
};
__global__ __launch_bounds__(512) void k_flow256_adj_reduce(const float* __restrict__ small, int gs,
                                                            const float* __restrict__ dw, int gd, AdjOut O) {
  __shared__ double R[8][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int y = blockIdx.y;                       // 0: small, 1, 2: dW1, dW2
  const int len = y == 0 ? kAdjSmall : kAdjDw, rows = y == 0 ? gs : gd;
  const int e = blockIdx.x * 64 + lane;
  if (blockIdx.x * 64 >= len) return;
  const float* p = y == 0 ? small : dw + (size_t)(y - 1) * gd * kAdjDw;
  double s = 0.0;
  if (e < len) {
#pragma unroll 4
    for (int b = w; b < rows; b += 8) s += p[(size_t)b * len + e];
  }
  R[w][lane] = s;
  __syncthreads();
  if (w || e >= len) return;
  double t = R[0][lane];
  for (int k = 1; k < 8; ++k) t += R[k][lane];
  const float v = (float)t;
  if (y == 0) {
    if (e < 3 * kH) O.W0[e] = v;
    else if (e < 4 * kH) O.b0[e - 3 * kH] = v;
    else if (e < 7 * kH) O.W3[e - 4 * kH] = v;
    else O.b3[e - 7 * kH] = v;
  } else {
    float* W = y == 1 ? O.W1 : O.W2;
    float* b = y == 1 ? O.b1 : O.b2;
    if (e < kH * kH) W[e] = v;
    else b[e - kH * kH] = v;
  }
}

int cus() {
  int dev = 0, v = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0)
    v = 256;
  return v;
}
// one workgroup per CU, none with less than a 32-point block
int grid_points(int64_t n) { return (int)std::min<int64_t>((n + 31) / 32, cus()); }
// half the CUs for each of the two products, at least 8 chunks of 32 stage points each
int grid_dw(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>((4 * n / 32 + 7) / 8, cus() / 2)); }

}  // namespace
}  // namespace mo

using namespace mo;

MO_EXPORT int mo_flow256_step_stages(const float* y0, int64_t n, const float* packed, float h, float* y1, float* Zs,
                                     void* stream) {
  MO_CHECK(packed && n >= 0 && n <= (1LL << 30) && (n == 0 || (y0 && y1)), MO_ERR_ARG,
           "mo_flow256_step_stages: bad arguments");
  MO_CHECK(((uintptr_t)packed & 15) == 0, MO_ERR_ARG, "mo_flow256_step_stages: packed not 16-byte aligned");
  if (n == 0) return MO_OK;
  hipLaunchKernelGGL(k_flow256_fwd, dim3(grid_points(n)), dim3(kThreads), 0, (hipStream_t)stream, y0, (int)n, packed,
                     h, y1, Zs);
  MO_HIP(hipGetLastError());
  return MO_OK;
}

MO_EXPORT int mo_flow256_step(const float* y0, int64_t n, const float* packed, float h, float* y1, void* stream) {
  MO_CHECK(packed && n >= 0 && n <= (1LL << 30) && (n == 0 || (y0 && y1)), MO_ERR_ARG,
           "mo_flow256_step: bad arguments");
  MO_CHECK(((uintptr_t)packed & 15) == 0, MO_ERR_ARG, "mo_flow256_step: packed not 16-byte aligned");
  if (n == 0) return MO_OK;
  hipLaunchKernelGGL(k_flow256_fwd, dim3(grid_points(n)), dim3(kThreads), 0, (hipStream_t)stream, y0, (int)n, packed,
                     h, y1, (float*)nullptr);
  MO_HIP(hipGetLastError());
  return MO_OK;
}

MO_EXPORT int64_t mo_flow256_adjoint_work_floats(int64_t n) {
  if (n <= 0) return 0;
  return 16 * kH * n + 2LL * grid_dw(n) * kAdjDw + (int64_t)grid_points(n) * kAdjSmall;
}

MO_EXPORT int mo_flow256_adjoint_step(int64_t n, const float* packed, float h, const float* Zs, const float* gy1,
                                      float* gy0, float* work, int32_t first, void* stream) {
  MO_CHECK(n > 0 && n <= (1LL << 25) && packed && Zs && gy1 && gy0 && work, MO_ERR_ARG,
           "mo_flow256_adjoint_step: bad arguments");
  MO_CHECK((((uintptr_t)packed | (uintptr_t)work) & 15) == 0, MO_ERR_ARG,
           "mo_flow256_adjoint_step: packed / work not 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  float* dw = work + 16 * kH * n;
  float* small = dw + 2LL * grid_dw(n) * kAdjDw;
  hipLaunchKernelGGL(k_flow256_adj, dim3(grid_points(n)), dim3(kThreads), 0, s, (int)n, packed, h, Zs, gy1, gy0, work,
                     small, first ? 1 : 0);
  hipLaunchKernelGGL(k_flow256_adj_dw, dim3(grid_dw(n), 2), dim3(kThreads), 0, s, (long long)4 * n, work, dw,
                     first ? 1 : 0);
  MO_HIP(hipGetLastError());
  return MO_OK;
}

MO_EXPORT int mo_flow256_adjoint_grads(int64_t n, const float* work, float* W0, float* b0, float* W1, float* b1,
                                       float* W2, float* b2, float* W3, float* b3, void* stream) {
  MO_CHECK(n > 0 && n <= (1LL << 30) / 12 && work && W0 && b0 && W1 && b1 && W2 && b2 && W3 && b3, MO_ERR_ARG,
           "mo_flow256_adjoint_grads: bad arguments");
  const float* dw = work + 16 * kH * n;
  hipLaunchKernelGGL(k_flow256_adj_reduce, dim3((kAdjDw + 63) / 64, 3), dim3(512), 0, (hipStream_t)stream,
                     dw + 2LL * grid_dw(n) * kAdjDw, grid_points(n), dw, grid_dw(n),
                     AdjOut{W0, b0, W1, b1, W2, b2, W3, b3});
  MO_HIP(hipGetLastError());
  return MO_OK;
}
