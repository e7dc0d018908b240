// Distance-field build: Mesh::ConstructDistanceField (mesh.cc:106-152) on
// gfx950, plus the template normalization (Mesh::Normalize, mesh.cc:66-96)
// and Mesh::ApplyTransform (mesh.cc:98-105) it depends on.
//
// Grid point (i, j, k) sits at (k/N, j/N, i/N) (mesh.cc:110-116) and its
// value is sqrt of the squared distance to the nearest target triangle
// (mesh.cc:140-150, igl::point_mesh_squared_distance).  The squared distance
// is computed in FP64 with a canonical operation sequence (face region when
// the projection falls inside, else the three edges with endpoints ordered
// by vertex index) so that triangles sharing an edge or vertex produce the
// identical value and ties resolve to the lowest triangle index.  This file
// is compiled with -ffp-contract=off: every FP64 operation is one IEEE
// rounding, so results are bit-reproducible on the host.
//
// Kernel structure (HBM traffic is small; the build is bound by VALU issue,
// 73% of the SIMDs' cycles for 512 box-union grids, the FP64 exact tests and
// the FP32 bounds about half each):
//   1. k_face_bins   : per face, index check + Morton bin of the centroid
//                      (16^3 bins).
//   2. k_bin_sort    : one workgroup counting-sorts face indices by bin (LDS
//                      histogram + scan) so tiles of consecutive faces are
//                      spatially tight.
//   3. k_face_prep   : FP64 face record and FP32 culling record per face,
//                      written in sorted order.
//   4. k_tile_bounds : AABB per tile of kTile (8) sorted faces and per
//                      super-tile of kSuperTiles (16) tiles.
//   5. k_grid_build  : one wavefront per 4x4x8 brick of grid points (two
//                      points per lane, 4 apart in z).  The
//                      wave first evaluates the 6 tiles nearest its brick's
//                      centre among the tiles of the 4 nearest super-tiles
//                      (they seed every lane with a near-exact distance),
//                      then walks the super-tiles 64 at a time: a
//                      brick-level ballot drops super-tiles whose AABB is
//                      farther from the brick than the wave's worst best
//                      distance, the tiles of the kept ones (64 per pass)
//                      go through the same test, and each remaining tile is
//                      kept only if some lane's own point-to-AABB bound
//                      still reaches that lane's best.  For a kept tile,
//                      one lane per face first drops the faces whose AABB
//                      is out of reach of the whole brick; the survivors'
//                      records are copied into LDS with coalesced loads,
//                      and the wave walks them (one LDS address for all
//                      lanes), testing a face exactly only when its AABB
//                      and plane bounds can still improve some lane.  Ties
//                      keep the lowest face index, so the visiting order
//                      never changes the result.
//   6. k_grid_heavy  : the bricks whose walk is long, again on 16 wavefronts
//                      each.
#include "mo_common.h"
#include "mo_grid.h"

#include <algorithm>
#include <cmath>
#include <vector>

namespace mo {

namespace {

// faces per culling tile: with the super-tile level below, 8 against 16
// gave 41.4 against 42.7 ms for 512 box-union grids at 64^3 (65 against
// 90 bound checks per cell: tighter tile AABBs) and the same time for the
// mixed 64^3 / 128^3 icosphere targets of up to 81,920 faces; 4 was
// slower (43.8 ms).  Without super-tiles 16 beat 32 and 8 (the scan over
// all tiles grew with their number).
constexpr int kTile = 8;
constexpr int kSeedTiles = 6;  // nearest tiles evaluated before the culled walk (4: 39.7, 8: 44.0 ms against 38.8)
// tiles per super-tile: the walk culls 128-face super-tiles against the
// brick first, then the tiles of the kept ones (four super-tiles, 64 tiles,
// per wavefront pass), so the walk's cost grows with the super-tiles near
// the brick rather than with the whole target (32 tiles per super-tile was
// slower: 47.7 ms, the seeds then come from two super-tiles)
constexpr int kSuperTiles = 16;
constexpr int kSupPass = 64 / kSuperTiles;   // super-tiles whose tiles one wavefront pass covers
static_assert(kSuperTiles * kSupPass == 64 && kSuperTiles <= 64, "a pass covers 64 tiles");
constexpr int kBinBits = 4;                  // 16 bins per axis
constexpr int kBins = 1 << (3 * kBinBits);   // 4096

__device__ inline unsigned spread3(unsigned v) {
  // spread the low 4 bits of v to every third bit
  unsigned r = 0;
  for (int b = 0; b < kBinBits; ++b) r |= ((v >> b) & 1u) << (3 * b);
  return r;
}

__device__ inline double dmin(double a, double b) { return b < a ? b : a; }
__device__ inline double dmax(double a, double b) { return b > a ? b : a; }
// One-instruction v_min_f64 for the minimum of the three edge distances: the
// operands are never NaN there, and where two operands are equal (including
// +0 / -0) either result gives the same comparisons.
__device__ inline double vmin(double a, double b) { return __builtin_fmin(a, b); }

// Pass 1: validate indices and compute the centroid bin (Morton order of a
// 16^3 lattice over [0,1]^3, clamped).  blockIdx.y = job.
__global__ void k_face_bins(const GridJob* __restrict__ jobs, int* __restrict__ err, GridQueue* __restrict__ queue) {
  const GridJob J = jobs[blockIdx.y];
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) queue->count = queue->next = 0;
  for (long long f = (long long)blockIdx.x * blockDim.x + threadIdx.x; f < J.nf;
       f += (long long)gridDim.x * blockDim.x) {
    double c[3] = {0.0, 0.0, 0.0};
    for (int j = 0; j < 3; ++j) {
      int vi = J.F[f * 3 + j];
      if (vi < 0 || vi >= J.nv) { atomicOr(err, 1); vi = 0; }
      for (int a = 0; a < 3; ++a) c[a] += J.V[(long long)vi * 3 + a];
    }
    unsigned b3[3];
    for (int a = 0; a < 3; ++a) {
      int b = (int)floor(c[a] * (1.0 / 3.0) * (1 << kBinBits));
      b = b < 0 ? 0 : (b > (1 << kBinBits) - 1 ? (1 << kBinBits) - 1 : b);
      b3[a] = (unsigned)b;
    }
    J.bin[f] = spread3(b3[0]) | (spread3(b3[1]) << 1) | (spread3(b3[2]) << 2);
  }
}

// Pass 2: one workgroup per job counting-sorts face indices by bin (LDS
// histogram, block-wide scan of the 4096 bins, LDS-atomic scatter).  The
// set-up kernels of a batch use workgroups of at most 256 threads (one
// wavefront per SIMD), which fit beside a running grid build's wavefronts,
// so a second batch's set-up is not held back behind them.
constexpr int kSortT = 256;
constexpr int kBinsPerThread = kBins / kSortT;   // 16 consecutive bins each
__global__ void __launch_bounds__(kSortT) k_bin_sort(const GridJob* __restrict__ jobs) {
  const GridJob J = jobs[blockIdx.x];
  __shared__ unsigned hist[kBins];
  __shared__ unsigned wsum[kSortT / 64];
  for (int b = threadIdx.x; b < kBins; b += blockDim.x) hist[b] = 0;
  __syncthreads();
  for (long long f = threadIdx.x; f < J.nf; f += blockDim.x) atomicAdd(&hist[J.bin[f]], 1u);
  __syncthreads();
  // exclusive scan: each thread owns kBinsPerThread consecutive bins
  const int t = threadIdx.x;
  unsigned v[kBinsPerThread];
  unsigned mine = 0;
#pragma unroll
  for (int q = 0; q < kBinsPerThread; ++q) {
    v[q] = hist[kBinsPerThread * t + q];
    mine += v[q];
  }
  unsigned incl = mine;
  const int lane = t & 63, w = t >> 6;
  for (int o = 1; o < 64; o <<= 1) {
    unsigned y = __shfl_up(incl, o, 64);
    if (lane >= o) incl += y;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  unsigned base = 0;
  for (int q = 0; q < w; ++q) base += wsum[q];
  unsigned ex = base + incl - mine;
#pragma unroll
  for (int q = 0; q < kBinsPerThread; ++q) {
    hist[kBinsPerThread * t + q] = ex;
    ex += v[q];
  }
  __syncthreads();
  for (long long f = threadIdx.x; f < J.nf; f += blockDim.x) {
    unsigned pos = atomicAdd(&hist[J.bin[f]], 1u);
    J.perm[pos] = (int)f;
  }
}

__device__ inline float round_down(double x) {
  const float f = (float)x;
  return (double)f > x ? nextafterf(f, -INFINITY) : f;
}
__device__ inline float round_up(double x) {
  const float f = (float)x;
  return (double)f < x ? nextafterf(f, INFINITY) : f;
}

// Pass 3: FP64 face record of face perm[pos] and its FP32 culling record,
// written at its sorted position.
// At most 64 VGPRs and one wavefront per SIMD and workgroup, so that a second
// batch's face preparation gets in when wavefronts of the first one's grid
// build (95 VGPRs, 5 per SIMD) or solver end, and not only when those kernels
// do.  (Two batches of 512 pairs in flight, 61 ms each: it takes 13 to 20 ms
// instead of 0.5.)
__global__ void __launch_bounds__(256, 8) k_face_prep(const GridJob* __restrict__ jobs) {
  const GridJob J = jobs[blockIdx.y];
  const double* __restrict__ V = J.V;
  const int* __restrict__ F = J.F;
  const long long nv = J.nv;
  for (long long pos = (long long)blockIdx.x * blockDim.x + threadIdx.x; pos < J.nf;
       pos += (long long)gridDim.x * blockDim.x) {
  const long long f = J.perm[pos];
  GFace g;
  int idx[3];
  double p[3][3];
  for (int j = 0; j < 3; ++j) {
    int vi = F[f * 3 + j];
    if (vi < 0 || vi >= nv) vi = 0;     // reported by k_face_bins
    idx[j] = vi;
    p[j][0] = V[(long long)vi * 3 + 0];
    p[j][1] = V[(long long)vi * 3 + 1];
    p[j][2] = V[(long long)vi * 3 + 2];
  }
  g.ax = p[0][0]; g.ay = p[0][1]; g.az = p[0][2];
  g.bx = p[1][0]; g.by = p[1][1]; g.bz = p[1][2];
  g.cx = p[2][0]; g.cy = p[2][1]; g.cz = p[2][2];
  double e0x = g.bx - g.ax, e0y = g.by - g.ay, e0z = g.bz - g.az;
  double e1x = g.cx - g.ax, e1y = g.cy - g.ay, e1z = g.cz - g.az;
  g.nx = e0y * e1z - e0z * e1y;
  g.ny = e0z * e1x - e0x * e1z;
  g.nz = e0x * e1y - e0y * e1x;
  double nn = g.nx * g.nx + g.ny * g.ny + g.nz * g.nz;
  g.inv_nn = nn > 0.0 ? 1.0 / nn : 0.0;
  g.d00 = e0x * e0x + e0y * e0y + e0z * e0z;
  g.d01 = e0x * e1x + e0y * e1y + e0z * e1z;
  g.d11 = e1x * e1x + e1y * e1y + e1z * e1z;
  g.denom = g.d00 * g.d11 - g.d01 * g.d01;
  int flip = 0;
  double ll[3], il[3];
  for (int j = 0; j < 3; ++j) {
    int i0 = j, i1 = (j + 1) % 3;
    if (idx[i1] < idx[i0]) { flip |= 1 << j; int t = i0; i0 = i1; i1 = t; }
    double dx = p[i1][0] - p[i0][0], dy = p[i1][1] - p[i0][1], dz = p[i1][2] - p[i0][2];
    ll[j] = dx * dx + dy * dy + dz * dz;
    il[j] = ll[j] > 0.0 ? 1.0 / ll[j] : 0.0;
  }
  g.ll0 = ll[0]; g.ll1 = ll[1]; g.ll2 = ll[2];
  g.il0 = il[0]; g.il1 = il[1]; g.il2 = il[2];
  g.flip = flip;
  g.face = (int)f;
  J.faces[pos] = g;
  GCull q;
  q.lox = round_down(dmin(g.ax, dmin(g.bx, g.cx))); q.hix = round_up(dmax(g.ax, dmax(g.bx, g.cx)));
  q.loy = round_down(dmin(g.ay, dmin(g.by, g.cy))); q.hiy = round_up(dmax(g.ay, dmax(g.by, g.cy)));
  q.loz = round_down(dmin(g.az, dmin(g.bz, g.cz))); q.hiz = round_up(dmax(g.az, dmax(g.bz, g.cz)));
  q.nx = q.ny = q.nz = q.c = q.e = q.pad = 0.f;
  // FP32 error of n . q - c for |q_i| <= 1: 3 products and sums of terms
  // below 3 + |c|, their operands rounded to 2^-24: under 1e-6 (1 + |c|).
  // n itself is good to 1e-9 where the triangle's sine exceeds 1e-6, and c
  // sums terms as large as the coordinates m: 1e-9 m more, which counts
  // where a face's vertices lie far from the box that its plane crosses.
  if (nn > 1e-12 * g.d00 * g.d11) {
    const double inv = 1.0 / sqrt(nn);
    const double ux = g.nx * inv, uy = g.ny * inv, uz = g.nz * inv;
    const double c = ux * g.ax + uy * g.ay + uz * g.az;
    q.nx = (float)ux; q.ny = (float)uy; q.nz = (float)uz;
    q.c = (float)c;
    const double m = dmax(dmax(dmax(-(double)q.lox, (double)q.hix), dmax(-(double)q.loy, (double)q.hiy)),
                          dmax(-(double)q.loz, (double)q.hiz));
    q.e = (float)(1e-6 * (1.0 + (c < 0.0 ? -c : c)) + 1e-9 * m);
  }
  J.cull[pos] = q;
  }
}

// One thread per tile: the union of its faces' AABBs; the 16 lanes of a
// super-tile then combine theirs.  (A wavefront per tile took 1.6 ms for 512
// targets of 9952 faces.)
__global__ void __launch_bounds__(256) k_tile_bounds(const GridJob* __restrict__ jobs) {
  const GridJob J = jobs[blockIdx.y];
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  float v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
  const long long f1 = (t + 1) * kTile < J.nf ? (t + 1) * kTile : J.nf;
  for (long long f = t * kTile; f < f1; ++f) {
    const float* g = &J.cull[f].lox;
    for (int a = 0; a < 3; ++a) {
      v[a] = fminf(v[a], g[a]);
      v[3 + a] = fmaxf(v[3 + a], g[3 + a]);
    }
  }
  if (t < J.ntiles)
    for (int a = 0; a < 6; ++a) J.tb[t * 6 + a] = v[a];
  for (int o = 1; o < kSuperTiles; o <<= 1)
    for (int a = 0; a < 3; ++a) {
      v[a] = fminf(v[a], __shfl_xor(v[a], o, 64));
      v[3 + a] = fmaxf(v[3 + a], __shfl_xor(v[3 + a], o, 64));
    }
  const long long sp = t / kSuperTiles;
  if (sp < J.nsuper && (t & (kSuperTiles - 1)) == 0)
    for (int a = 0; a < 6; ++a) J.sb[sp * 6 + a] = v[a];
}

// Canonical edge squared distance (endpoints ordered by vertex index).
__device__ inline double edge_d2(double qx, double qy, double qz, double ux, double uy, double uz,
                                 double wx, double wy, double wz, double ll, double il) {
  double dx = wx - ux, dy = wy - uy, dz = wz - uz;
  double px = qx - ux, py = qy - uy, pz = qz - uz;
  double tn = px * dx + py * dy + pz * dz;
  if (tn <= 0.0 || ll == 0.0) return px * px + py * py + pz * pz;
  if (tn >= ll) {
    double rx = qx - wx, ry = qy - wy, rz = qz - wz;
    return rx * rx + ry * ry + rz * rz;
  }
  double t = tn * il;
  double cx = ux + t * dx, cy = uy + t * dy, cz = uz + t * dz;
  double rx = qx - cx, ry = qy - cy, rz = qz - cz;
  return rx * rx + ry * ry + rz * rz;
}

__device__ inline double face_d2(const GFace& g, double qx, double qy, double qz) {
  double vx = qx - g.ax, vy = qy - g.ay, vz = qz - g.az;
  if (g.denom > 0.0 && g.inv_nn > 0.0) {
    double e0x = g.bx - g.ax, e0y = g.by - g.ay, e0z = g.bz - g.az;
    double e1x = g.cx - g.ax, e1y = g.cy - g.ay, e1z = g.cz - g.az;
    double d20 = vx * e0x + vy * e0y + vz * e0z;
    double d21 = vx * e1x + vy * e1y + vz * e1z;
    double bb = g.d11 * d20 - g.d01 * d21;
    double cc = g.d00 * d21 - g.d01 * d20;
    if (bb >= 0.0 && cc >= 0.0 && bb + cc <= g.denom) {
      double dp = g.nx * vx + g.ny * vy + g.nz * vz;
      return (dp * dp) * g.inv_nn;
    }
  }
  // edge j joins p_j and p_{j+1}; flip bit j set when p_{j+1} has the lower
  // index.  The face is the same in every lane, so the flip bits are read
  // into a scalar register and each edge takes one uniform branch.
  const int flip = __builtin_amdgcn_readfirstlane(g.flip);
  double d0, d1, d2;
  if (flip & 1) d0 = edge_d2(qx, qy, qz, g.bx, g.by, g.bz, g.ax, g.ay, g.az, g.ll0, g.il0);
  else d0 = edge_d2(qx, qy, qz, g.ax, g.ay, g.az, g.bx, g.by, g.bz, g.ll0, g.il0);
  if (flip & 2) d1 = edge_d2(qx, qy, qz, g.cx, g.cy, g.cz, g.bx, g.by, g.bz, g.ll1, g.il1);
  else d1 = edge_d2(qx, qy, qz, g.bx, g.by, g.bz, g.cx, g.cy, g.cz, g.ll1, g.il1);
  if (flip & 4) d2 = edge_d2(qx, qy, qz, g.ax, g.ay, g.az, g.cx, g.cy, g.cz, g.ll2, g.il2);
  else d2 = edge_d2(qx, qy, qz, g.cx, g.cy, g.cz, g.ax, g.ay, g.az, g.ll2, g.il2);
  return vmin(vmin(d2, d1), d0);
}

// Device memory reached through the job table's pointers: the explicit
// global address space makes the accesses global_* instead of flat_*
// instructions (a flat load also counts against the LDS wait counter, so
// every LDS wait would wait for it).
#if defined(__HIP_DEVICE_COMPILE__)
#define MO_GLOBAL __attribute__((address_space(1)))
#else
#define MO_GLOBAL
#endif
template <class T>
__device__ inline MO_GLOBAL T* gptr(T* p) {
  return (MO_GLOBAL T*)p;
}

// Wave-wide reductions through DPP lane moves (quad_perm [1,0,3,2] and
// [2,3,0,1], row_half_mirror, row_mirror), then the four row results by
// readlane: every lane gets the same value, with no LDS permutes.
template <int CTRL>
__device__ inline unsigned dpp_u32(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}
template <int CTRL>
__device__ inline float dpp_f32(float v) {
  return __uint_as_float(dpp_u32<CTRL>(__float_as_uint(v)));
}
__device__ inline float readlane_f32(float v, int l) {
  return __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(v), l));
}
__device__ inline float wave_max(float v) {
  v = fmaxf(v, dpp_f32<0xB1>(v));
  v = fmaxf(v, dpp_f32<0x4E>(v));
  v = fmaxf(v, dpp_f32<0x141>(v));
  v = fmaxf(v, dpp_f32<0x140>(v));
  return fmaxf(fmaxf(readlane_f32(v, 0), readlane_f32(v, 16)), fmaxf(readlane_f32(v, 32), readlane_f32(v, 48)));
}
__device__ inline unsigned wave_min_u32(unsigned v) {
  v = min(v, dpp_u32<0xB1>(v));
  v = min(v, dpp_u32<0x4E>(v));
  v = min(v, dpp_u32<0x141>(v));
  v = min(v, dpp_u32<0x140>(v));
  const unsigned a = (unsigned)__builtin_amdgcn_readlane((int)v, 0), b = (unsigned)__builtin_amdgcn_readlane((int)v, 16),
                 c = (unsigned)__builtin_amdgcn_readlane((int)v, 32), d = (unsigned)__builtin_amdgcn_readlane((int)v, 48);
  return min(min(a, b), min(c, d));
}
// the lane holding the (nearly) smallest non-negative key, -1 when every
// lane is out: the low bits of the key give way to the lane number
__device__ inline int nearest_lane(float key, bool in) {
  const unsigned k = in ? (__float_as_uint(key) & ~63u) | (threadIdx.x & 63u) : 0xFFFFFFFFu;
  const unsigned m = wave_min_u32(k);
  return m == 0xFFFFFFFFu ? -1 : (int)(m & 63u);
}

// Culling in FP32.  A lower bound of a squared distance is formed from
// outward-rounded AABBs; beside the real gap D it is at most
// (D + 5.2e-8)^2 (1 + 5e-7): the grid point's coordinates in [0, 1) are
// rounded by 2^-25 an axis, and the subtractions and fused sums by 2^-24
// relative.  cut_of(best) is above that for every D <= sqrt(best), so a
// bound beyond it shows that the face can neither improve nor tie the best.
// (FP64 bounds, 18 operations without contraction where FP32 needs 11, on
// records of twice the size: 36.7 ms against 31.2 for 512 box-union grids.)
__device__ inline float cut_of(double best) {
  const float r = __builtin_sqrtf((float)best) * 1.000002f + 2e-7f;
  return r * r * 1.000002f;
}
__device__ inline float gap1(float lo, float hi, float a, float b) {   // [lo, hi] against [a, b]
  return fmaxf(fmaxf(lo - b, a - hi), 0.f);
}
__device__ inline float box_gap2(const MO_GLOBAL float* __restrict__ tb, long long t, float lx, float ly, float lz,
                                 float hx, float hy, float hz) {
  const MO_GLOBAL float* b = tb + t * 6;
  const float gx = gap1(b[0], b[3], lx, hx), gy = gap1(b[1], b[4], ly, hy), gz = gap1(b[2], b[5], lz, hz);
  return __builtin_fmaf(gz, gz, __builtin_fmaf(gy, gy, gx * gx));
}

// LDS of one wavefront: the survivors of a tile's brick-level cull, culling
// records and full records
struct WaveTile {
  GFace face[kTile];
  float4 cull[3 * kTile];
  int list[kTile];
};
// orders a wavefront's own LDS accesses (the hardware keeps their order)
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

constexpr int kZPts = 2;          // points per lane, 4 apart in z
constexpr int kHeavyWaves = 16;   // wavefronts of a brick in the second kernel

// LDS the wavefronts of one brick share in the second kernel
struct BrickShare {
  unsigned cut[kZPts][64];                  // culling thresholds, FP32 bits (non-negative: integer order)
  double best[kHeavyWaves][kZPts][64];
  int idx[kHeavyWaves][kZPts][64];
};

// One 4x4x8 brick: lane l holds the two grid points (x, y, z) and
// (x, y, z + 4) of it.  The two points share the brick's culling, the staged
// face records, every LDS read of a record and the x / y parts of their
// bounds.  With kWaves > 1 the tiles are dealt out to the wavefronts by their
// number, every wavefront holding all points; they share their culling
// thresholds through LDS and merge their bests at the end.  With one
// wavefront, a brick that has walked max_tiles tiles is given up (false).
template <int kWaves>
__device__ inline bool grid_brick(const GridJob& JJ, int b, int max_tiles, WaveTile& L, BrickShare* S) {
  const MO_GLOBAL GFace* __restrict__ faces = gptr(JJ.faces);
  const MO_GLOBAL GCull* __restrict__ cull = gptr(JJ.cull);
  const long long nf = JJ.nf;
  const MO_GLOBAL float* __restrict__ tb = gptr(JJ.tb);
  const long long ntiles = JJ.ntiles;
  const MO_GLOBAL float* __restrict__ sb = gptr(JJ.sb);
  const long long nsuper = JJ.nsuper;
  const int N = JJ.N;
  const int bpa = (N + 3) / 4;
  MO_GLOBAL double* __restrict__ dist64 = gptr(JJ.dist64);
  MO_GLOBAL float* __restrict__ dist32 = gptr(JJ.dist32);
  MO_GLOBAL int* __restrict__ nearest = gptr(JJ.nearest);
  const int lane = threadIdx.x & 63, wv = kWaves > 1 ? (int)(threadIdx.x >> 6) : 0;
  const int bx = b % bpa;
  const int by = (b / bpa) % bpa;
  const int bz = b / (bpa * bpa);
  const int k = bx * 4 + (lane & 3), j = by * 4 + ((lane >> 2) & 3);
  int ip[kZPts];
  bool valid[kZPts];
  double qz[kZPts];
  const double qx = (double)k / (double)N, qy = (double)j / (double)N;
  float fz[kZPts];
  const float fx = (float)qx, fy = (float)qy;
#pragma unroll
  for (int s = 0; s < kZPts; ++s) {
    ip[s] = bz * 4 * kZPts + (lane >> 4) + 4 * s;
    valid[s] = (k < N) && (j < N) && (ip[s] < N);
    qz[s] = (double)ip[s] / (double)N;
    fz[s] = (float)qz[s];
  }
  // brick AABB over valid points
  const int k1 = min(bx * 4 + 3, N - 1), j1 = min(by * 4 + 3, N - 1), i1 = min(bz * 4 * kZPts + 4 * kZPts - 1, N - 1);
  const float lx = (float)((double)(bx * 4) / N), ly = (float)((double)(by * 4) / N),
              lz = (float)((double)(bz * 4 * kZPts) / N);
  const float hx = (float)((double)k1 / N), hy = (float)((double)j1 / N), hz = (float)((double)i1 / N);

  // points farther than the band only need to be shown farther (GridSpec);
  // cut: the FP32 culling threshold kept with best (-1: no point here, below
  // every bound)
  double best[kZPts];
  float cut[kZPts];
  int bidx[kZPts];
#pragma unroll
  for (int s = 0; s < kZPts; ++s) {
    best[s] = JJ.band2;
    cut[s] = valid[s] ? cut_of(best[s]) : -1.f;
    bidx[s] = INT_MAX;
  }
  if (kWaves > 1) {
    if (wv == 0)
#pragma unroll
      for (int s = 0; s < kZPts; ++s) S->cut[s][lane] = __float_as_uint(valid[s] ? cut[s] : 0.f);
    __syncthreads();
  }
  // the thresholds the brick's other wavefronts have reached
  auto refresh = [&]() {
    if (kWaves > 1)
#pragma unroll
      for (int s = 0; s < kZPts; ++s)
        if (valid[s]) cut[s] = fminf(cut[s], __uint_as_float(*(volatile unsigned*)&S->cut[s][lane]));
  };
  // the wave's worst threshold over its valid points
  auto worst = [&]() { return wave_max(fmaxf(cut[0], cut[1])); };
  static_assert(kZPts == 2, "worst() takes two points");
  // work counters (wave-uniform): exact evaluations (one point per lane),
  // lanes that needed one, face bound checks (per point), staged tiles
  unsigned long long n_exact = 0, n_needed = 0, n_bound = 0, n_tiles = 0;

  // bound: an upper bound of every valid point's threshold (the wave's worst
  // when it was taken; thresholds only shrink, so an older value stays valid)
  auto process_tile = [&](int t, float bound) {
    const long long f0 = (long long)t * kTile;
    const int cnt = (int)((nf - f0) < kTile ? (nf - f0) : kTile);
    // stage 1, one face per lane: drop faces whose AABB is farther from the
    // brick AABB than the wave's worst best distance
    bool cand = false;
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    f32x4 c0, c1, c2;
    if (lane < cnt) {
      const MO_GLOBAL f32x4* gp = reinterpret_cast<const MO_GLOBAL f32x4*>(cull + f0 + lane);
      c0 = gp[0]; c1 = gp[1]; c2 = gp[2];
      const float ax = gap1(c0.x, c0.w, lx, hx), ay = gap1(c0.y, c1.x, ly, hy), az = gap1(c0.z, c1.y, lz, hz);
      cand = !(__builtin_fmaf(az, az, __builtin_fmaf(ay, ay, ax * ax)) > bound);
    }
    const unsigned long long m = __ballot(cand);
    const int ns = __popcll(m);
    if (ns == 0) return;
    ++n_tiles;
    n_bound += (unsigned long long)ns * kZPts;
    // compact the survivors (in face order) and stage their records in LDS
    const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
    wave_sync();   // the last tile's records have been read
    if (cand) {
      L.list[rank] = lane;
      f32x4* d = reinterpret_cast<f32x4*>(L.cull) + 3 * rank;
      d[0] = c0; d[1] = c1; d[2] = c2;
    }
    wave_sync();
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    constexpr int kChunks = (int)(sizeof(GFace) / sizeof(u32x4));
    static_assert(sizeof(GFace) % sizeof(u32x4) == 0 && sizeof(GCull) == 48, "records are copied in 16-byte chunks");
    const MO_GLOBAL u32x4* __restrict__ src = reinterpret_cast<const MO_GLOBAL u32x4*>(faces + f0);
    u32x4* dst = reinterpret_cast<u32x4*>(L.face);
    for (int c = lane; c < ns * kChunks; c += 64) {
      const int r = c / kChunks, w = c - r * kChunks;
      dst[c] = src[L.list[r] * kChunks + w];
    }
    wave_sync();
    refresh();
    // stage 2, per surviving face: every point's own AABB bound, then (when
    // it leaves some point) the plane bound, then the exact test when some
    // lane's point can still improve or tie its best
    for (int r = 0; r < ns; ++r) {
      const float4 r0 = L.cull[3 * r], r1 = L.cull[3 * r + 1], r2 = L.cull[3 * r + 2];
      const float gx = gap1(r0.x, r0.w, fx, fx), gy = gap1(r0.y, r1.x, fy, fy);
      const float gxy = __builtin_fmaf(gy, gy, gx * gx);
      bool mine[kZPts];
      bool any = false;
#pragma unroll
      for (int s = 0; s < kZPts; ++s) {
        const float gz = gap1(r0.z, r1.y, fz[s], fz[s]);
        mine[s] = !(__builtin_fmaf(gz, gz, gxy) > cut[s]);
        any = any || mine[s];
      }
      if (!__ballot(any)) continue;
      // the face plane is a second lower bound
      const float dxy = __builtin_fmaf(r1.z, fx, __builtin_fmaf(r1.w, fy, -r2.y));
#pragma unroll
      for (int s = 0; s < kZPts; ++s) {
        const float dp = fmaxf(fabsf(__builtin_fmaf(r2.x, fz[s], dxy)) - r2.z, 0.f);
        mine[s] = mine[s] && !(dp * dp > cut[s]);
      }
#pragma unroll
      for (int s = 0; s < kZPts; ++s) {
        const unsigned long long need = __ballot(mine[s]);
        if (!need) continue;
        ++n_exact;
        n_needed += (unsigned long long)__popcll(need);
        // only the lanes that need it evaluate (a point whose bound exceeds
        // its best cannot improve or tie it), so the face-region / edge
        // branches diverge over those lanes alone
        if (mine[s]) {
          const GFace& g = L.face[r];
          const double d = face_d2(g, qx, qy, qz[s]);
          if (d < best[s] || (d == best[s] && g.face < bidx[s])) {
            best[s] = d;
            cut[s] = fminf(cut[s], cut_of(d));
            bidx[s] = g.face;
            if (kWaves > 1) atomicMin(&S->cut[s][lane], __float_as_uint(cut[s]));
          }
        }
      }
    }
  };

  // 1. seeds: the kSupPass super-tiles nearest to the brick's centre (one
  //    scan of the super-tile AABBs; each lane keeps its nearest), then the
  //    kSeedTiles nearest of their 64 tiles, are evaluated first.  They give
  //    every point a near-exact distance, which makes the culling below
  //    tight (the choice of seeds affects speed only).
  int seedv = -1, nseed = 0;   // lane r holds the r-th seed
  {
    // ranked by the AABB gap from the brick's centre (a brick inside
    // several AABBs has gap 0 to all of them)
    const float cx = 0.5f * (lx + hx), cy = 0.5f * (ly + hy), cz = 0.5f * (lz + hz);
    float slb = INFINITY;
    int ss = -1;
    for (long long c = 0; c < nsuper; c += 64) {
      const long long sidx = c + lane;
      if (sidx >= nsuper) continue;
      const float lb = box_gap2(sb, sidx, cx, cy, cz, cx, cy, cz);
      if (lb < slb) { slb = lb; ss = (int)sidx; }
    }
    int sp[kSupPass];
    for (int u = 0; u < kSupPass; ++u) sp[u] = -1;
    for (int u = 0; u < kSupPass; ++u) {
      const int at = nearest_lane(slb, ss >= 0);
      if (at < 0) break;
      sp[u] = __builtin_amdgcn_readlane(ss, at);
      if (lane == at) ss = -1;
    }
    const int q = lane / kSuperTiles;
    int sq = -1;
#pragma unroll
    for (int u = 0; u < kSupPass; ++u) sq = q == u ? sp[u] : sq;
    float mlb = INFINITY;
    int mt = -1;
    if (sq >= 0) {
      const long long t = (long long)sq * kSuperTiles + (lane & (kSuperTiles - 1));
      if (t < ntiles) {
        mlb = box_gap2(tb, t, cx, cy, cz, cx, cy, cz);
        mt = (int)t;
      }
    }
    for (int r = 0; r < kSeedTiles; ++r) {
      const int at = nearest_lane(mlb, mt >= 0);
      if (at < 0) break;
      const int st = __builtin_amdgcn_readlane(mt, at);
      if (lane == r) seedv = st;
      ++nseed;
      if (lane == at) mt = -1;
    }
  }

  // 2. every other tile that can still improve (or tie) some point's best:
  //    super-tiles whose AABB is within the wave's worst best of the brick
  //    AABB, then (kSupPass kept super-tiles per pass, lane kSuperTiles q + j
  //    on tile j of the q-th) their tiles by the same test, and each such
  //    tile is kept only if some point's own point-to-AABB bound reaches its
  //    own best.
  //    (One loop for both, so that the face tests are compiled in once.)
  int walked = 0, seed = 0;
  long long c = 0, t = -1;
  unsigned long long smask = 0, tmask = 0;
  float bound = 0.f;
  while (true) {
    int tt;
    if (seed < nseed) {
      const int r = seed++;
      if (kWaves > 1 && r % kWaves != wv) continue;
      tt = __builtin_amdgcn_readlane(seedv, r);
      bound = worst();
    } else {
      if (seed == nseed) {      // after the seeds
        ++seed;
        if (kWaves > 1) __syncthreads();
      }
      if (!tmask) {
        refresh();
        bound = worst();
        if (!smask) {
          if (c >= nsuper) break;
          const long long sidx = c + lane;
          const float slb = sidx < nsuper ? box_gap2(sb, sidx, lx, ly, lz, hx, hy, hz) : INFINITY;
          smask = __ballot(sidx < nsuper && !(slb > bound));
          c += 64;
          if (!smask) continue;
        }
        const long long first = c - 64;
        const int q = lane / kSuperTiles;
        int sq = -1;
#pragma unroll
        for (int u = 0; u < kSupPass; ++u) {
          const int sp = smask ? (int)first + __ffsll((long long)smask) - 1 : -1;
          smask &= smask - 1;
          sq = q == u ? sp : sq;
        }
        t = sq < 0 ? -1 : (long long)sq * kSuperTiles + (lane & (kSuperTiles - 1));
        bool need = false;
        if (t >= 0 && t < ntiles && (kWaves == 1 || (lane & (kWaves - 1)) == wv))
          need = !(box_gap2(tb, t, lx, ly, lz, hx, hy, hz) > bound);
#pragma unroll
        for (int r = 0; r < kSeedTiles; ++r) need = need && __builtin_amdgcn_readlane(seedv, r) != (int)t;
        tmask = __ballot(need);
        continue;
      }
      const int l = __ffsll((long long)tmask) - 1;
      tmask &= tmask - 1;
      tt = __builtin_amdgcn_readlane((int)t, l);
      const MO_GLOBAL float* tbb = tb + (long long)tt * 6;
      const float gx = gap1(tbb[0], tbb[3], fx, fx), gy = gap1(tbb[1], tbb[4], fy, fy);
      const float gxy = __builtin_fmaf(gy, gy, gx * gx);
      bool reach = false;
#pragma unroll
      for (int s = 0; s < kZPts; ++s) {
        const float gz = gap1(tbb[2], tbb[5], fz[s], fz[s]);
        reach = reach || !(__builtin_fmaf(gz, gz, gxy) > cut[s]);
      }
      if (!__ballot(reach)) continue;
      if (kWaves == 1 && ++walked > max_tiles) return false;
    }
    process_tile(tt, bound);
  }
  static_assert(kWaves == 1 || kSuperTiles % kWaves == 0, "tiles are dealt by their number in a super-tile");
  if (JJ.stats && lane == 0) {
    atomicAdd(JJ.stats + kGridStatExact, n_exact * 64ull);
    atomicAdd(JJ.stats + kGridStatExactNeeded, n_needed);
    atomicAdd(JJ.stats + kGridStatBound, n_bound * 64ull);
    atomicAdd(JJ.stats + kGridStatTiles, n_tiles);
  }
  if (kWaves > 1) {
#pragma unroll
    for (int s = 0; s < kZPts; ++s) {
      S->best[wv][s][lane] = best[s];
      S->idx[wv][s][lane] = bidx[s];
    }
    __syncthreads();
    if (wv == 0)
#pragma unroll
      for (int s = 0; s < kZPts; ++s)
        for (int w = 1; w < kWaves; ++w) {
          const double d = S->best[w][s][lane];
          const int i = S->idx[w][s][lane];
          if (d < best[s] || (d == best[s] && i < bidx[s])) { best[s] = d; bidx[s] = i; }
        }
    __syncthreads();   // the next brick overwrites the shared arrays
    if (wv != 0) return true;
  }
#pragma unroll
  for (int s = 0; s < kZPts; ++s) {
    if (!valid[s]) continue;
    const long long cell = ((long long)ip[s] * N + j) * N + k;
    const double sq = sqrt(best[s]);
    if (dist64) dist64[cell] = sq;
    if (dist32) dist32[cell] = (float)sq;
    if (nearest) nearest[cell] = bidx[s] == INT_MAX ? -1 : bidx[s];
  }
  return true;
}

__device__ inline int brick_count(int N) {
  const int bpa = (N + 3) / 4, bpz = (N + 4 * kZPts - 1) / (4 * kZPts);
  return bpa * bpa * bpz;
}

// One wavefront per brick.  Most bricks walk a few tiles; one near the
// target's medial surface can walk hundreds (1400 of a 81,920-face sphere at
// 128^3, 8.4 ms, where the median brick takes 37 us), and a launch of few
// bricks lasts as long as its worst.  A brick past max_tiles goes to the
// queue (which holds every brick), and k_grid_heavy starts it again on 16
// wavefronts.
__global__ void __launch_bounds__(64, 5) k_grid_build(const GridJob* __restrict__ jobs, GridQueue* __restrict__ queue,
                                                   int max_tiles) {
  __shared__ WaveTile L;
  const GridJob& JJ = jobs[blockIdx.y];
  const int b = blockIdx.x;
  if (b >= brick_count(JJ.N)) return;
  if (grid_brick<1>(JJ, b, max_tiles, L, nullptr)) return;
  if (threadIdx.x == 0) queue->item[atomicAdd(&queue->count, 1)] = make_int2((int)blockIdx.y, b);
}

__global__ void __launch_bounds__(64 * kHeavyWaves) k_grid_heavy(const GridJob* __restrict__ jobs,
                                                                 GridQueue* __restrict__ queue) {
  __shared__ WaveTile L[kHeavyWaves];
  __shared__ BrickShare S;
  __shared__ int s_item;
  const int n = queue->count;
  while (true) {
    if (threadIdx.x == 0) s_item = atomicAdd(&queue->next, 1);
    __syncthreads();
    const int q = s_item;
    if (q >= n) return;
    const int2 it = queue->item[q];
    grid_brick<kHeavyWaves>(jobs[it.x], it.y, INT_MAX, L[threadIdx.x >> 6], &S);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Normalization (Mesh::Normalize, mesh.cc:66-96) on device, FP64.

__device__ inline double xf_read(const XformJob& J, long long i) {
  return J.f64 ? ((const double*)J.V)[i] : (double)((const float*)J.V)[i];
}

// One workgroup per job: min / max per axis, then scale and pos (exact
// whatever the workgroup size: minima and maxima do not round).
constexpr int kStatT = 256;
__global__ void __launch_bounds__(kStatT) k_normalize_stats(const XformJob* __restrict__ jobs) {
  const XformJob J = jobs[blockIdx.x];
  __shared__ double smn[3][kStatT], smx[3][kStatT];
  double mn[3] = {1e30, 1e30, 1e30}, mx[3] = {-1e30, -1e30, -1e30};
  for (long long i = threadIdx.x; i < J.n; i += blockDim.x)
    for (int a = 0; a < 3; ++a) {
      double v = xf_read(J, i * 3 + a);
      if (v < mn[a]) mn[a] = v;
      if (v > mx[a]) mx[a] = v;
    }
  for (int a = 0; a < 3; ++a) { smn[a][threadIdx.x] = mn[a]; smx[a][threadIdx.x] = mx[a]; }
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s)
      for (int a = 0; a < 3; ++a) {
        double o = smn[a][threadIdx.x + s];
        if (o < smn[a][threadIdx.x]) smn[a][threadIdx.x] = o;
        o = smx[a][threadIdx.x + s];
        if (o > smx[a][threadIdx.x]) smx[a][threadIdx.x] = o;
      }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double ex = smx[0][0] - smn[0][0], ey = smx[1][0] - smn[1][0], ez = smx[2][0] - smn[2][0];
    double m = ez > ey ? ez : ey;           // std::max(b, c)
    m = m > ex ? m : ex;                    // std::max(a, .)
    double scale = m * 1.1;
    J.sp[0] = scale;
    for (int a = 0; a < 3; ++a) J.sp[1 + a] = smn[a][0] - 0.05 * scale;
  }
}

// out = (V - pos) / scale with the job's (scale, pos); blockIdx.y = job.
__global__ void k_apply_transform(const XformJob* __restrict__ jobs) {
  const XformJob J = jobs[blockIdx.y];
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < J.n * 3;
       i += (long long)gridDim.x * blockDim.x) {
    int a = (int)(i % 3);
    J.out[i] = (xf_read(J, i) - J.sp[1 + a]) / J.sp[0];
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// Host launchers.

static size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

size_t grid_job_workspace_bytes(long long nf) {
  const long long ntiles = (nf + kTile - 1) / kTile;
  const long long nsuper = (ntiles + kSuperTiles - 1) / kSuperTiles;
  return al256((size_t)nf * sizeof(GFace)) + al256((size_t)nf * sizeof(GCull)) + al256((size_t)nf * sizeof(unsigned)) +
         al256((size_t)nf * sizeof(int)) + al256((size_t)ntiles * 6 * sizeof(float)) +
         al256((size_t)nsuper * 6 * sizeof(float));
}

static long long brick_total(long long N) {
  const long long bpa = (N + 3) / 4, bpz = (N + 4 * kZPts - 1) / (4 * kZPts);
  return bpa * bpa * bpz;
}
static size_t queue_bytes(long long bricks) { return al256(sizeof(GridQueue) + (size_t)bricks * sizeof(int2)); }

int grid_check_resolution(int N) {
  MO_CHECK(N >= 2 && N <= 2048, MO_ERR_ARG, "grid resolution %d out of range [2, 2048]", N);
  return MO_OK;
}

int grid_build_batch_launch(const GridSpec* specs, int n, void* workspace, hipStream_t stream, int* err_dev,
                            hipEvent_t build_after) {
  if (n <= 0) return MO_OK;
  std::vector<GridJob> jobs(n);
  char* w = (char*)workspace;
  GridJob* d_jobs = (GridJob*)w;
  w += al256((size_t)n * sizeof(GridJob));
  long long bricks = 0;
  for (int q = 0; q < n; ++q) {
    if (int rc = grid_check_resolution(specs[q].N)) return rc;
    bricks += brick_total(specs[q].N);
  }
  GridQueue* queue = (GridQueue*)w;
  w += queue_bytes(bricks);
  long long max_nf = 0, max_tiles = 0, max_bricks = 0;
  for (int q = 0; q < n; ++q) {
    const GridSpec& sp = specs[q];
    MO_CHECK(sp.nf >= 1, MO_ERR_ARG, "distance field needs at least one triangle (got %lld)", sp.nf);
    GridJob& J = jobs[q];
    J.V = sp.Vn; J.F = sp.F; J.nv = sp.nv; J.nf = sp.nf; J.N = sp.N;
    J.ntiles = (sp.nf + kTile - 1) / kTile;
    J.faces = (GFace*)w; w += al256((size_t)sp.nf * sizeof(GFace));
    J.cull = (GCull*)w; w += al256((size_t)sp.nf * sizeof(GCull));
    J.bin = (unsigned*)w; w += al256((size_t)sp.nf * sizeof(unsigned));
    J.perm = (int*)w; w += al256((size_t)sp.nf * sizeof(int));
    J.tb = (float*)w; w += al256((size_t)J.ntiles * 6 * sizeof(float));
    J.nsuper = (J.ntiles + kSuperTiles - 1) / kSuperTiles;
    J.sb = (float*)w; w += al256((size_t)J.nsuper * 6 * sizeof(float));
    J.dist64 = sp.dist64; J.dist32 = sp.dist32; J.nearest = sp.nearest;
    MO_CHECK(sp.band2 > 0.0, MO_ERR_ARG, "grid band must be positive");
    J.band2 = sp.band2;
    J.stats = sp.stats;
    max_nf = std::max(max_nf, sp.nf);
    max_tiles = std::max(max_tiles, J.ntiles);
    max_bricks = std::max(max_bricks, brick_total(sp.N));
  }
  int rc = chain_h2d(d_jobs, jobs.data(), (size_t)n * sizeof(GridJob), stream);
  if (rc) return rc;
  const int T = 256;
  const unsigned fb = (unsigned)std::min<long long>((max_nf + T - 1) / T, 1024);
  hipLaunchKernelGGL(k_face_bins, dim3(fb, n), dim3(T), 0, stream, d_jobs, err_dev, queue);
  hipLaunchKernelGGL(k_bin_sort, dim3(n), dim3(kSortT), 0, stream, d_jobs);
  hipLaunchKernelGGL(k_face_prep, dim3(fb, n), dim3(T), 0, stream, d_jobs);
  hipLaunchKernelGGL(k_tile_bounds, dim3((unsigned)((max_tiles + 255) / 256), n), dim3(256), 0, stream, d_jobs);
  if (build_after) MO_HIP(hipStreamWaitEvent(stream, build_after, 0));
  // Where a brick is handed over: the tail matters the more the fewer bricks
  // share the chip, the work done twice the more the more there are: a
  // multiple of the square root of the launch's bricks (34 tiles for one 64^3
  // grid, 96 for one 128^3 grid, 768 for 512 64^3 grids).  Multiples 0.5,
  // 0.75, 1: one 5000-vertex box target at 64^3 0.48, 0.49, 0.54 ms, a
  // 2562-vertex sphere at 50^3 0.78, 0.85, 0.92, a 642-vertex pair 2.76, 2.81,
  // 2.84, a 10242-vertex sphere at 128^3 5.12, 4.92, 4.60, 48 mixed pairs
  // 76.1, 74.7, 73.8: small launches want less, large ones more.  0.25, 2 and
  // 4 are behind on one side or both, and so are 4 or 8 wavefronts in the
  // second kernel.
  const int max_tiles_brick = std::max(16, (int)(0.75 * std::sqrt((double)bricks)));
  hipLaunchKernelGGL(k_grid_build, dim3((unsigned)max_bricks, n), dim3(64), 0, stream, d_jobs, queue,
                     max_tiles_brick);
  hipLaunchKernelGGL(k_grid_heavy, dim3((unsigned)std::min<long long>(512, bricks)), dim3(64 * kHeavyWaves), 0, stream,
                     d_jobs, queue);
  MO_HIP(hipGetLastError());
  return MO_OK;
}

size_t grid_batch_workspace_bytes(const GridSpec* specs, int n) {
  size_t b = al256((size_t)n * sizeof(GridJob));
  long long bricks = 0;
  for (int q = 0; q < n; ++q) {
    b += grid_job_workspace_bytes(specs[q].nf);
    bricks += brick_total(specs[q].N);
  }
  return b + queue_bytes(bricks) + 256;
}

size_t xform_workspace_bytes(int n) { return al256((size_t)n * sizeof(XformJob)) + 256; }

int xform_batch_launch(const XformJob* jobs, int n, bool compute_stats, void* workspace, hipStream_t stream) {
  if (n <= 0) return MO_OK;
  XformJob* d_jobs = (XformJob*)workspace;
  long long max_n = 0;
  for (int q = 0; q < n; ++q) max_n = std::max(max_n, jobs[q].n);
  int rc = chain_h2d(d_jobs, jobs, (size_t)n * sizeof(XformJob), stream);
  if (rc) return rc;
  if (compute_stats) hipLaunchKernelGGL(k_normalize_stats, dim3(n), dim3(kStatT), 0, stream, d_jobs);
  if (max_n > 0) {
    const unsigned bx = (unsigned)std::min<long long>((max_n * 3 + 255) / 256, 1024);
    hipLaunchKernelGGL(k_apply_transform, dim3(bx, n), dim3(256), 0, stream, d_jobs);
  }
  MO_HIP(hipGetLastError());
  return MO_OK;
}

}  // namespace mo
