// Register/LDS-resident variant of the batched LM solver (same algorithm as
// mo_lm.hip: Deformer::Deform / DeformGraph, deformer.cc:18-92, 370-442,
// with Ceres' trust-region LM restated and a matrix-free block-Jacobi PCG).
//
// One workgroup of T threads solves one pair whose nv <= T * VPT vertices
// are statically owned (vertex i by thread i % T, slot i / T).  Everything
// the PCG iterates on lives in VGPRs for the whole solve: the distance
// gradient g, the direction p, q = A p, the step delta and
// d = lambda^2 deg + LM diagonal / radius (the diagonal of A apart from
// g g^T, which is also the block-Jacobi preconditioner's diagonal).  The
// one vector neighbours read (u while evaluating the Jacobian, z = M^-1 r
// inside PCG, u + delta for the candidate) is published to a
// float4-per-vertex LDS array whose w holds the vertex's adjacency word
// (LDS offset << 16 | count) for the whole solve; the PCG residual is not
// stored but recovered as r = M z from the published z.  The pair's
// adjacency is copied once into LDS as uint16 entries (neighbour << 1 |
// multiplicity - 1), each vertex's list padded to even length with a zero
// vector slot so the PCG product reads two entries per 32-bit word; pairs
// whose entries all share one multiplicity skip the per-entry weight.  The
// PCG loop touches no global memory.  Reductions are FP64, through DPP lane
// moves and one LDS exchange between waves.
//
// Differences from the global kernel that do not change the algorithm:
//   * the preconditioner M = g g^T + diag(d) is applied with the
//     Sherman-Morrison formula each iteration instead of a stored inverse;
//   * A p is formed as A z + beta A p_prev (p = z + beta p_prev), so only z
//     is published and an iteration needs two barriers;
//   * the rigidity residuals are linear in x, so the rigidity part of the
//     model cost change equals its actual change E_r(u + delta) - E_r(u);
//     only u + delta has to be gathered for the candidate.
#include "mo_common.h"
#include "mo_lm.h"
#include "mo_lm_util.h"
#include "mo_lookup.h"

#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <string>
#include <vector>

namespace mo {

namespace {

// global slots of LMArrays::work used here; gOrder: a large pair's spatial
// order (int perm[nv], inv[nv] and the sort's scratch), gSlots: a pair's
// TagTeam words
enum GSlot { gGR = 1, gS = 2, gDG = 3, gZ = 4, gOrder = 5, gSlots = 6 };
static_assert(gSlots < kLMWorkSlots, "work slots");

// Block-wide exclusive scan of one int per thread (T <= 1024).
__device__ inline int block_exclusive_scan(int x, int* buf, int& total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  int v = x;
  for (int o = 1; o < 64; o <<= 1) {
    int t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  if (lane == 63) buf[w] = v;
  __syncthreads();
  int base = 0;
  total = 0;
  for (int q = 0; q < nw; ++q) {
    if (q < w) base += buf[q];
    total += buf[q];
  }
  __syncthreads();
  return base + v - x;
}

// x, y, z of an LDS vertex record (w, the vertex's adjacency word, stays).
typedef float mo_v3f __attribute__((ext_vector_type(3)));
__device__ inline void store_xyz(float4* p, float4 v) {
  mo_v3f t;
  t.x = v.x; t.y = v.y; t.z = v.z;
  *reinterpret_cast<mo_v3f*>(p) = t;
}

// A solve after a rejected step starts from that step (scaled) instead of
// from zero (see solve below).
constexpr bool kPcgWarmStart = true;

// An index the optimizer cannot see through: per-vertex addresses are then
// formed at each use (base + index) instead of being hoisted out of the
// solver loops, where they would hold dozens of registers for the whole
// kernel.
__device__ inline int opaque(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// First record of a halo team's copies of neighbours: behind the own
// vertices and behind the set-up's bitmap (a bit per vertex of the pair and
// a 16-bit count per word).
__host__ __device__ inline int halo_base(int own, int nv) {
  const int words = (nv + 31) / 32, overlay = (words * 6 + 15) / 16;
  return own > overlay ? own : overlay;
}

// The solver body, shared by the one-workgroup kernel (LdsSolo: all nv
// vertices in the workgroup's LDS array), the halo team (LdsHalo: a
// workgroup owns a range of the pair's vertices and keeps copies of the
// neighbours outside it behind them, read from the pair's publication array
// once per publication) and the team for meshes whose
// halo does not fit (LdsTeam: every access to such a neighbour reads the
// publication array).  Entry: an adjacency entry type (uint16 local indices,
// uint32 pair indices for LdsTeam).
template <int T, int VPT, class Team, class Entry>
__device__ inline void lds_solve(const LMPairDesc& P, int pid, Team& team, const LMArrays& A,
                                 const LMOptionsDev& opt, LMResultDev* __restrict__ res, long long totalV,
                                 unsigned char* smem, double* red, int* scan_buf, unsigned lds_bytes) {
  const double o_min_diag = opt.min_lm_diagonal, o_max_diag = opt.max_lm_diagonal;
  const float o_pcg_tol = opt.pcg_relative_tolerance;
  const bool o_pcg_warm = kPcgWarmStart;
  const int o_pcg_max = opt.pcg_max_iterations;
  const int tid = threadIdx.x;
  const int own = team.hi - team.lo;       // owned vertices: local index t + k T < own
  const long long vb = P.vbase;
  const float l2 = P.lambda * P.lambda;
  const float* __restrict__ grid = P.grid;
  const int N = P.N;
  const float4* __restrict__ X0 = A.x0 + vb;
  float4* __restrict__ U = A.u + vb;
  const int2* __restrict__ ADJ = A.adj + vb;
  const unsigned* __restrict__ NB = A.nbr + P.ebase;
  float4* __restrict__ GR = A.work + (size_t)gGR * totalV + vb;
  float4* __restrict__ S = A.work + (size_t)gS * totalV + vb;
  float4* __restrict__ DG = A.work + (size_t)gDG * totalV + vb;
  float4* __restrict__ ZG = A.work + (size_t)gZ * totalV + vb;   // team: published vectors
  // paired layout: a zero vector behind the vertex records, and every
  // vertex's entry list padded to even length with it, so the PCG product
  // reads two entries per 32-bit LDS word
  constexpr bool kPaired = Team::kPaired;
  float4* VEC = (float4*)smem;             // own vertices at their local index, then a halo team's copies of neighbours
  int sel = 0;
  const long long clock_start = wall_clock64();

  // ---- adjacency -> LDS (packed, compacted by a block scan) -------------
  // each own vertex's (LDS offset << 16) | count lives in VEC[il].w for the
  // whole solve (publications write x, y, z only), so it costs no register
  float uniform_m = 0.f;   // paired layout: the pair's multiplicity when all entries share it, else 0
  Entry* LCSR;
  {
    int cnt[VPT], gst[VPT], mine = 0;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int il = opaque(tid + k * T);
      cnt[k] = 0;
      gst[k] = 0;
      if (il < own) {
        const int2 a = ADJ[team.index(il)];
        gst[k] = a.x;
        cnt[k] = a.y;
        mine += kPaired ? a.y + (a.y & 1) : a.y;
      }
    }
    if constexpr (Team::kHalo) {
      // distinct neighbours owned elsewhere: a bitmap over the pair's ranks
      // (at the LDS' start, dead before the own records are written), its
      // words' prefix counts, and each one's rank in the w of its record
      unsigned* bm = (unsigned*)smem;
      const int nwords = (P.nv + 31) >> 5;
      unsigned short* pre = (unsigned short*)(bm + nwords);
      if ((size_t)halo_base(own, P.nv) * sizeof(float4) > lds_bytes) {
        team.give_up();
        return;
      }
      for (int q = tid; q < nwords; q += blockDim.x) bm[q] = 0u;
      __syncthreads();
#pragma unroll
      for (int k = 0; k < VPT; ++k)
        for (int e = 0; e < cnt[k]; ++e) {
          const int q = team.rank(nb_index(NB[gst[k] + e]));
          if ((unsigned)(q - team.lo) < (unsigned)own) continue;
          team.shared |= 1u << k;
          atomicOr(&bm[q >> 5], 1u << (q & 31));
        }
      __syncthreads();
      const int per = (nwords + (int)blockDim.x - 1) / (int)blockDim.x;
      const int q0 = min(nwords, tid * per), q1 = min(nwords, q0 + per);
      int bits = 0;
      for (int q = q0; q < q1; ++q) bits += __popc(bm[q]);
      int nh;
      int h = block_exclusive_scan(bits, scan_buf, nh);
      team.nhalo = nh;
      team.hbase = halo_base(own, P.nv);
      for (int q = q0; q < q1; ++q) {
        pre[q] = (unsigned short)h;
        const int n = __popc(bm[q]);
        if ((size_t)(team.hbase + h + n) * sizeof(float4) <= lds_bytes) {
          int r = team.hbase + h;
          for (unsigned m = bm[q]; m; m &= m - 1) reinterpret_cast<int*>(VEC + r++)[3] = q * 32 + __ffs((int)m) - 1;
        }
        h += n;
      }
      __syncthreads();
    }
    const int zero = team.hbase + team.nhalo;   // the zero vector's index
    const int records = zero + (kPaired ? 1 : 0);
    LCSR = (Entry*)(smem + (size_t)records * sizeof(float4));
    int total;
    int off = block_exclusive_scan(mine, scan_buf, total);
    // the launch's LDS was sized from the same adjacency; a mismatch (a
    // replayed graph whose inputs' faces changed) leaves the pair unsolved
    // and is reported by the host, never written past the allocation
    if ((size_t)records * sizeof(float4) + (size_t)total * sizeof(Entry) > lds_bytes ||
        (Team::kHalo && (records > 32767 || total > 65535))) {
      team.give_up();
      return;
    }
    int has1 = 0, has2 = 0;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      int o = off;
      for (int e = 0; e < cnt[k]; ++e, ++o) {
        const unsigned en = NB[gst[k] + e];
        has1 |= (en >> 24) == 1u;
        has2 |= (en >> 24) == 2u;
        int j = team.rank(nb_index(en));
        if constexpr (Team::kHalo) {
          if ((unsigned)(j - team.lo) < (unsigned)own) {
            j -= team.lo;
          } else {
            const unsigned* bm = (const unsigned*)smem;
            const unsigned short* pre = (const unsigned short*)(bm + ((P.nv + 31) >> 5));
            j = team.hbase + (int)pre[j >> 5] + __popc(bm[j >> 5] & ((1u << (j & 31)) - 1u));
          }
        }
        LCSR[o] = (Entry)(((unsigned)j << 1) | ((en >> 24) - 1u));
      }
      if (kPaired && (cnt[k] & 1)) LCSR[o] = (Entry)((unsigned)zero << 1);
      off += kPaired ? cnt[k] + (cnt[k] & 1) : cnt[k];
    }
    if constexpr (Team::kHalo) __syncthreads();   // the bitmap is dead from here
    off -= mine;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int il = opaque(tid + k * T);
      if (il < own) reinterpret_cast<float*>(VEC + il)[3] = __uint_as_float(((unsigned)off << 16) | (unsigned)cnt[k]);
      off += kPaired ? cnt[k] + (cnt[k] & 1) : cnt[k];
    }
    if constexpr (kPaired) {
      int any1 = __syncthreads_or(has1), any2 = __syncthreads_or(has2);
      if constexpr (Team::kHalo) {
        double any[2] = {any1 ? 1.0 : 0.0, any2 ? 1.0 : 0.0};
        team.template reduce<0, 2>(any, red, sel);
        any1 = any[0] > 0.0;
        any2 = any[1] > 0.0;
      }
      uniform_m = any1 && !any2 ? 1.f : (any2 && !any1 ? 2.f : 0.f);
      if (tid == 0) VEC[zero] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }

  // ---- per-vertex register state ----------------------------------------
  // g: distance gradient; p: direction; q = A p; d = lambda^2 deg + LM
  // diagonal / radius (the diagonal of A without g g^T, also the
  // preconditioner's diagonal); e: the step delta.  The PCG residual r is
  // not stored: r = M z for the z = M^-1 r held in LDS.
  float gx[VPT], gy[VPT], gz[VPT];
  float px[VPT], py[VPT], pz[VPT];
  float qx[VPT], qy[VPT], qz[VPT];
  float dx[VPT], dy[VPT], dz[VPT];
  float ex[VPT], ey[VPT], ez[VPT];

  // z = M^-1 r with M = g g^T + diag(d) (Sherman-Morrison)
  auto precond = [&](int k, float r0, float r1, float r2, float& z0, float& z1, float& z2) {
    const float i0 = __builtin_amdgcn_rcpf(dx[k]), i1 = __builtin_amdgcn_rcpf(dy[k]),
                i2 = __builtin_amdgcn_rcpf(dz[k]);
    const float h0 = gx[k] * i0, h1 = gy[k] * i1, h2 = gz[k] * i2;
    const float sig = 1.0f + gx[k] * h0 + gy[k] * h1 + gz[k] * h2;
    const float c = (h0 * r0 + h1 * r1 + h2 * r2) * __builtin_amdgcn_rcpf(sig);
    z0 = r0 * i0 - h0 * c;
    z1 = r1 * i1 - h1 * c;
    z2 = r2 * i2 - h2 * c;
  };

  // sum over the vertex's neighbours of multiplicity * VEC[neighbour].xyz
  auto gather = [&](int cs, float& sx, float& sy, float& sz) {
    sx = 0.f; sy = 0.f; sz = 0.f;
    const int o = (int)((unsigned)cs >> 16), c = cs & 0xFFFF;
    if constexpr (kPaired) {
      // two entries per LDS word (offsets are even; an odd list ends with
      // the zero slot), two independent neighbour reads in flight
      const unsigned* __restrict__ L2 = reinterpret_cast<const unsigned*>(LCSR) + (o >> 1);
      const int n2 = (c + 1) >> 1;
      // (the entry indices pass through opaque() so each address is one
      // bit-field extract and one shift-add)
      const unsigned* const L2e = L2 + n2;
      if (uniform_m != 0.f) {
        #pragma unroll 1
        for (const unsigned* pw = L2; pw < L2e; ++pw) {
          const unsigned w = *pw;
          const float4 a = VEC[opaque((int)__builtin_amdgcn_ubfe(w, 1, 15))];
          const float4 b = VEC[opaque((int)__builtin_amdgcn_ubfe(w, 17, 15))];
          if constexpr (Team::kInOrder) {
            sx += a.x; sy += a.y; sz += a.z;
            sx += b.x; sy += b.y; sz += b.z;
          } else {
            sx += a.x + b.x; sy += a.y + b.y; sz += a.z + b.z;
          }
        }
        sx *= uniform_m; sy *= uniform_m; sz *= uniform_m;
      } else {
        #pragma unroll 1
        for (const unsigned* pw = L2; pw < L2e; ++pw) {
          const unsigned w = *pw;
          const float4 a = VEC[opaque((int)__builtin_amdgcn_ubfe(w, 1, 15))];
          const float4 b = VEC[opaque((int)__builtin_amdgcn_ubfe(w, 17, 15))];
          const float ma = (float)((w & 1u) + 1u), mb = (float)(((w >> 16) & 1u) + 1u);
          if constexpr (Team::kInOrder) {
            sx += ma * a.x; sy += ma * a.y; sz += ma * a.z;
            sx += mb * b.x; sy += mb * b.y; sz += mb * b.z;
          } else {
            sx += ma * a.x + mb * b.x; sy += ma * a.y + mb * b.y; sz += ma * a.z + mb * b.z;
          }
        }
      }
    } else {
      #pragma unroll 1
      for (int q = 0; q < c; ++q) {
        const unsigned w = LCSR[o + q];
        const float m = (float)((w & 1u) + 1u);
        const float4 vj = team.neighbour(VEC, ZG, w >> 1);
        sx += m * vj.x; sy += m * vj.y; sz += m * vj.z;
      }
    }
  };

  auto eval = [&](bool first, double& cv, double& ce, double& gmax) {
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int il = opaque(tid + k * T);
      if (il < own) team.publish(VEC, ZG, k, il, U[team.index(il)]);
    }
    team.sync(VEC, ZG);
    double v[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int il = opaque(tid + k * T);
      if (il >= own) continue;
      const int i = team.index(il);
      const float4 x0 = X0[i];
      const float4 ui = VEC[il];
      const int cs = __float_as_int(ui.w);
      const JetF J = lookup_value_grad(grid, N, x0.x + ui.x, x0.y + ui.y, x0.z + ui.z);
      gx[k] = J.v0; gy[k] = J.v1; gz[k] = J.v2;
      const float ldk = l2 * x0.w;
      float sx = 0.f, sy = 0.f, sz = 0.f;
      double e = 0.0;
      const int o = (int)((unsigned)cs >> 16), c = cs & 0xFFFF;
      #pragma unroll 1
      for (int q = 0; q < c; ++q) {
        const unsigned w = LCSR[o + q];
        const float m = (float)((w & 1u) + 1u);
        const float4 uj = team.neighbour(VEC, ZG, w >> 1);
        const float ax = ui.x - uj.x, ay = ui.y - uj.y, az = ui.z - uj.z;
        sx += m * ax; sy += m * ay; sz += m * az;
        e += (double)m * ((double)ax * ax + (double)ay * ay + (double)az * az);
      }
      const float g0 = J.a * J.v0 + l2 * sx, g1 = J.a * J.v1 + l2 * sy, g2 = J.a * J.v2 + l2 * sz;
      GR[i] = make_float4(g0, g1, g2, J.a);   // J^T f and the residual d
      v[0] += 0.5 * (double)J.a * (double)J.a;
      v[1] += 0.25 * (double)l2 * e;
      double gm = fabs((double)g0);
      gm = fabs((double)g1) > gm ? fabs((double)g1) : gm;
      gm = fabs((double)g2) > gm ? fabs((double)g2) : gm;
      v[2] = gm > v[2] ? gm : v[2];
      if (first) {
        const float c0 = J.v0 * J.v0 + ldk, c1 = J.v1 * J.v1 + ldk, c2 = J.v2 * J.v2 + ldk;
        S[i] = make_float4(1.0f / (1.0f + sqrtf(c0)), 1.0f / (1.0f + sqrtf(c1)), 1.0f / (1.0f + sqrtf(c2)), 0.f);
      }
    }
    team.template reduce<2, 1>(v, red, sel);
    cv = v[0]; ce = v[1]; gmax = v[2];
  };

  // PCG on (J^T J + D^2 / radius) delta = -J^T f.  Each iteration publishes
  // z = M^-1 r once and forms A p as A z + beta A p_prev (p = z + beta
  // p_prev), so an iteration has two barriers: the reduction of p.Ap, and
  // the reduction of r.z and r.r, which also publishes the new z.
  //
  // After a rejected step (reuse: the same J^T J and J^T f, only the LM
  // diagonal grew) the solve starts from the rejected step e scaled by
  // alpha = (b . A e) / (e . A e), the best multiple of it in the A-norm,
  // instead of from zero; the stopping test stays |r| <= tol |b|, the same
  // absolute accuracy as a solve started from zero.
  auto solve = [&](bool reuse, double radius) -> int {
    const float finv_radius = (float)(1.0 / radius);
    const bool warm = reuse && o_pcg_warm;
    double v[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int il = opaque(tid + k * T);
      px[k] = py[k] = pz[k] = 0.f;
      qx[k] = qy[k] = qz[k] = 0.f;
      if (!warm) ex[k] = ey[k] = ez[k] = 0.f;
      dx[k] = dy[k] = dz[k] = 1.f;
      if (il >= own) continue;
      const int i = team.index(il);
      const float4 s = S[i];
      const float ldk = l2 * X0[i].w;
      float4 dg;
      if (!reuse) {
        const double cc[3] = {(double)gx[k] * gx[k] + ldk, (double)gy[k] * gy[k] + ldk,
                              (double)gz[k] * gz[k] + ldk};
        const double sc[3] = {s.x, s.y, s.z};
        float d3[3];
        for (int a = 0; a < 3; ++a) {
          double t = sc[a] * sc[a] * cc[a];
          t = t < o_min_diag ? o_min_diag : (t > o_max_diag ? o_max_diag : t);
          d3[a] = (float)t;
        }
        dg = make_float4(d3[0], d3[1], d3[2], 0.f);
        DG[i] = dg;
      } else {
        dg = DG[i];
      }
      // LM regularization D^2 / radius in the unscaled variables (the
      // diagonal over s^2), capped at 1e30; FP32 with a reciprocal (the
      // FP64 divisions' temporaries would set the kernel's register peak)
      dx[k] = ldk + fminf(dg.x * __builtin_amdgcn_rcpf(s.x * s.x) * finv_radius, 1e30f);
      dy[k] = ldk + fminf(dg.y * __builtin_amdgcn_rcpf(s.y * s.y) * finv_radius, 1e30f);
      dz[k] = ldk + fminf(dg.z * __builtin_amdgcn_rcpf(s.z * s.z) * finv_radius, 1e30f);
      if (warm) {
        team.publish(VEC, ZG, k, il, make_float4(ex[k], ey[k], ez[k], 0.f));
        continue;
      }
      const float4 gr = GR[i];
      const float r0 = -gr.x, r1 = -gr.y, r2 = -gr.z;
      float z0, z1, z2;
      precond(k, r0, r1, r2, z0, z1, z2);
      team.publish(VEC, ZG, k, il, make_float4(z0, z1, z2, 0.f));
      v[0] += (double)(r0 * z0 + r1 * z1 + r2 * z2);
      v[1] += (double)(r0 * r0 + r1 * r1 + r2 * r2);
    }
    if (warm) {
      // A e (into q) and the scaling alpha
      team.sync(VEC, ZG);
      double a2[2] = {0.0, 0.0};
#pragma unroll
      for (int k = 0; k < VPT; ++k) {
        const int il = opaque(tid + k * T);
        if (il >= own) continue;
        const float4 ei = VEC[il];
        float sx, sy, sz;
        gather(__float_as_int(ei.w), sx, sy, sz);
        const float gee = gx[k] * ei.x + gy[k] * ei.y + gz[k] * ei.z;
        qx[k] = gx[k] * gee + dx[k] * ei.x - l2 * sx;
        qy[k] = gy[k] * gee + dy[k] * ei.y - l2 * sy;
        qz[k] = gz[k] * gee + dz[k] * ei.z - l2 * sz;
        const float4 gr = GR[team.index(il)];
        a2[0] -= (double)(gr.x * qx[k] + gr.y * qy[k] + gr.z * qz[k]);
        a2[1] += (double)(ex[k] * qx[k] + ey[k] * qy[k] + ez[k] * qz[k]);
      }
      team.template reduce<2, 0>(a2, red, sel);
      const float al = a2[1] > 0.0 ? (float)(a2[0] / a2[1]) : 0.f;
#pragma unroll
      for (int k = 0; k < VPT; ++k) {
        const int il = opaque(tid + k * T);
        if (il >= own) continue;
        ex[k] *= al; ey[k] *= al; ez[k] *= al;
        const float4 gr = GR[team.index(il)];
        const float r0 = -gr.x - al * qx[k], r1 = -gr.y - al * qy[k], r2 = -gr.z - al * qz[k];
        qx[k] = qy[k] = qz[k] = 0.f;
        float z0, z1, z2;
        precond(k, r0, r1, r2, z0, z1, z2);
        team.publish(VEC, ZG, k, il, make_float4(z0, z1, z2, 0.f));
        v[0] += (double)(r0 * z0 + r1 * z1 + r2 * z2);
        v[1] += (double)(r0 * r0 + r1 * r1 + r2 * r2);
        v[2] += (double)(gr.x * gr.x + gr.y * gr.y + gr.z * gr.z);
      }
    }
    team.template reduce<3, 0>(v, red, sel);
    team.refresh(VEC, ZG);   // z is published
    double rz = v[0];
    const double rr0 = warm ? v[2] : v[1];     // |b|^2
    if (!(rr0 > 0.0)) return 0;
    const double tol2 = (double)o_pcg_tol * o_pcg_tol * rr0;
    if (warm && v[1] <= tol2) return 0;
    float beta = 0.f;
    int it = 0;
    while (it < o_pcg_max) {
      double w1[1] = {0.0};
#pragma unroll
      for (int k = 0; k < VPT; ++k) {
        const int il = opaque(tid + k * T);
        if (il >= own) continue;
        const float4 zi = VEC[il];
        float sx, sy, sz;
        gather(__float_as_int(zi.w), sx, sy, sz);
        const float gzz = gx[k] * zi.x + gy[k] * zi.y + gz[k] * zi.z;
        const float wx = gx[k] * gzz + dx[k] * zi.x - l2 * sx;
        const float wy = gy[k] * gzz + dy[k] * zi.y - l2 * sy;
        const float wz = gz[k] * gzz + dz[k] * zi.z - l2 * sz;
        px[k] = zi.x + beta * px[k]; py[k] = zi.y + beta * py[k]; pz[k] = zi.z + beta * pz[k];
        qx[k] = wx + beta * qx[k]; qy[k] = wy + beta * qy[k]; qz[k] = wz + beta * qz[k];
        w1[0] += (double)(px[k] * qx[k] + py[k] * qy[k] + pz[k] * qz[k]);
      }
      team.template reduce<1, 0>(w1, red, sel);
      const double pq = w1[0];
      if (!(pq > 0.0)) break;
      const float fa = (float)(rz / pq);
      double w2[2] = {0.0, 0.0};
#pragma unroll
      for (int k = 0; k < VPT; ++k) {
        const int il = opaque(tid + k * T);
        if (il >= own) continue;
        ex[k] += fa * px[k]; ey[k] += fa * py[k]; ez[k] += fa * pz[k];
        // the residual is not kept: r = M z for the z still published
        // (M = g g^T + diag(d), the preconditioner), then r -= alpha q
        const float4 zo = VEC[il];
        const float gzo = gx[k] * zo.x + gy[k] * zo.y + gz[k] * zo.z;
        const float r0 = gx[k] * gzo + dx[k] * zo.x - fa * qx[k];
        const float r1 = gy[k] * gzo + dy[k] * zo.y - fa * qy[k];
        const float r2 = gz[k] * gzo + dz[k] * zo.z - fa * qz[k];
        float z0, z1, z2;
        precond(k, r0, r1, r2, z0, z1, z2);
        team.publish(VEC, ZG, k, il, make_float4(z0, z1, z2, 0.f));
        w2[0] += (double)(r0 * z0 + r1 * z1 + r2 * z2);
        w2[1] += (double)(r0 * r0 + r1 * r1 + r2 * r2);
      }
      team.template reduce<2, 0>(w2, red, sel);
      ++it;
      if (w2[1] <= tol2) break;
      team.refresh(VEC, ZG);   // z is published
      beta = (float)(w2[0] / rz);
      rz = w2[0];
    }
    return it;
  };

  double ce_now = 0.0;   // rigidity energy at the current x (set by eval)
  auto candidate = [&]() -> LMCandidate {
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int il = opaque(tid + k * T);
      if (il < own) {
        const float4 ui = U[team.index(il)];
        team.publish(VEC, ZG, k, il, make_float4(ui.x + ex[k], ui.y + ey[k], ui.z + ez[k], 0.f));
      }
    }
    team.sync(VEC, ZG);
    double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int il = opaque(tid + k * T);
      if (il >= own) continue;
      const int i = team.index(il);
      const float4 x0 = X0[i];
      const float dres = GR[i].w;
      const float gd = gx[k] * ex[k] + gy[k] * ey[k] + gz[k] * ez[k];
      v[0] += (double)gd * ((double)dres + 0.5 * (double)gd);
      const float4 wv = VEC[il];
      const int cs = __float_as_int(wv.w);
      const float wx = wv.x, wy = wv.y, wz = wv.z;
      const float dc = lookup_f32(grid, N, x0.x + wx, x0.y + wy, x0.z + wz);
      v[1] += 0.5 * (double)dc * (double)dc;
      double e = 0.0;
      const int o = (int)((unsigned)cs >> 16), c = cs & 0xFFFF;
      #pragma unroll 1
      for (int q = 0; q < c; ++q) {
        const unsigned w = LCSR[o + q];
        const float m = (float)((w & 1u) + 1u);
        const float4 wj = team.neighbour(VEC, ZG, w >> 1);
        const float ax = wx - wj.x, ay = wy - wj.y, az = wz - wj.z;
        e += (double)m * ((double)ax * ax + (double)ay * ay + (double)az * az);
      }
      v[2] += 0.25 * (double)l2 * e;
      v[3] += (double)ex[k] * ex[k] + (double)ey[k] * ey[k] + (double)ez[k] * ez[k];
      const float4 ui = U[i];
      const float qx0 = x0.x + ui.x, qy0 = x0.y + ui.y, qz0 = x0.z + ui.z;
      v[4] += (double)qx0 * qx0 + (double)qy0 * qy0 + (double)qz0 * qz0;
    }
    team.template reduce<5, 0>(v, red, sel);
    // rigidity residuals are linear: their model change equals the actual one
    return LMCandidate{-v[0] - (v[2] - ce_now), v[1] + v[2], sqrt(v[3]), sqrt(v[4])};
  };

  auto eval_tracked = [&](bool first, double& cv, double& ce, double& gmax) {
    eval(first, cv, ce, gmax);
    ce_now = ce;
  };
  auto accept = [&]() {
    // u <- u + delta: exactly the candidate published to LDS
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int il = opaque(tid + k * T);
      if (il < own) {
        const float4 v = VEC[il];
        U[team.index(il)] = make_float4(v.x, v.y, v.z, 0.f);
      }
    }
  };
  lm_trust_region_loop(opt, eval_tracked, solve, candidate, accept, team.leader() ? res + pid : nullptr,
                       clock_start);
}

// One workgroup per pair.
struct LdsSolo {
  static constexpr bool kPaired = true, kHalo = false, kInOrder = false;
  int lo, hi, hbase, nhalo;
  __device__ explicit LdsSolo(int nv) : lo(0), hi(nv), hbase(nv), nhalo(0) {}
  __device__ bool leader() const { return true; }
  __device__ void give_up() {}
  __device__ int index(int il) const { return il; }
  __device__ int rank(int j) const { return j; }
  __device__ void sync(float4*, const float4*) { __syncthreads(); }
  __device__ void refresh(float4*, const float4*) {}
  template <int K, int M>
  __device__ void reduce(double (&v)[K + M], double* red, int& sel) { block_reduce_dpp<K, M>(v, red, sel); }
  __device__ float4 neighbour(const float4* VEC, const float4* ZG, unsigned j) const { return VEC[j]; }
  __device__ void publish(float4* VEC, float4* ZG, int k, int il, float4 v) const { store_xyz(VEC + il, v); }
};

// A team of workgroups per pair (co-resident: cooperative launch).
// Workgroup r owns [lo, hi).  The publication array ZG is written and read
// only through device-coherent stores and loads, and the team barrier and
// reductions are CoherentTeam's, so no barrier writes back or invalidates
// the L2.
struct LdsTeam {
  static constexpr bool kPaired = false, kHalo = false;
  CoherentTeam g;
  int lo, hi, hbase, nhalo;
  __device__ LdsTeam(const CoherentTeam& team, int l, int h) : g(team), lo(l), hi(h), hbase(h - l), nhalo(0) {}
  __device__ bool leader() const { return g.leader(); }
  __device__ void give_up() {}
  __device__ int index(int il) const { return lo + il; }
  __device__ int rank(int j) const { return j; }
  __device__ void sync(float4*, const float4*) { g.barrier(); }
  __device__ void refresh(float4*, const float4*) {}
  template <int K, int M>
  __device__ void reduce(double (&v)[K + M], double* red, int& sel) { g.template reduce_dpp<K, M>(v, red, sel); }
  __device__ float4 neighbour(const float4* VEC, const float4* ZG, unsigned j) const {
    const unsigned jl = j - (unsigned)lo;
    return jl < (unsigned)(hi - lo) ? VEC[jl] : load_coherent(ZG + j);
  }
  __device__ void publish(float4* VEC, float4* ZG, int k, int il, float4 v) const {
    store_xyz(VEC + il, v);
    store_coherent(ZG + lo + il, v);
  }
};

// A large pair's team: workgroup r owns the ranks [lo, hi) of the pair's
// vertices in the spatial order that k_chunk_plan made (perm: rank ->
// vertex, inv: vertex -> rank), which keeps halos short whatever the mesh's
// numbering.  Records hbase .. hbase + nhalo of VEC are copies of the
// neighbours owned elsewhere, each with its rank in w; only vertices that
// have such a neighbour (bit k of `shared` for slot k) are written to ZG,
// and refresh() copies the halo after the exchange that follows a
// publication.  A vertex's neighbours are then LDS reads as in LdsSolo:
// reading ZG in the gather cost a remote round trip per neighbour.
struct LdsHalo {
  static constexpr bool kPaired = true, kHalo = true, kInOrder = true;
  TagTeam g;
  int lo, hi, hbase, nhalo;
  unsigned shared;
  const int* perm;
  const int* inv;
  __device__ LdsHalo(const TagTeam& team, int l, int h, const int* p, const int* i)
      : g(team), lo(l), hi(h), hbase(h - l), nhalo(0), shared(0u), perm(p), inv(i) {}
  __device__ float4 neighbour(const float4* VEC, const float4* ZG, unsigned j) const { return VEC[j]; }
  __device__ void publish(float4* VEC, float4* ZG, int k, int il, float4 v) const {
    store_xyz(VEC + il, v);
    if (shared >> k & 1u) store_coherent(ZG + lo + il, v);
  }
  __device__ void refresh(float4* VEC, const float4* ZG) const {
    float4* rec = VEC + hbase;
    for (int h = threadIdx.x; h < nhalo; h += 2 * blockDim.x) {
      const int h2 = h + blockDim.x;
      const bool two = h2 < nhalo;
      const int r1 = reinterpret_cast<const int*>(rec + h)[3];
      const int r2 = two ? reinterpret_cast<const int*>(rec + h2)[3] : r1;
      const float4 a = load_coherent(ZG + r1), b = load_coherent(ZG + r2);
      store_xyz(rec + h, a);
      if (two) store_xyz(rec + h2, b);
    }
    __syncthreads();
  }
  __device__ bool leader() const { return g.leader(); }
  __device__ void give_up() { __hip_atomic_store(g.abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
  __device__ int index(int il) const { return perm[lo + il]; }
  __device__ int rank(int j) const { return inv[j]; }
  __device__ void sync(float4* VEC, const float4* ZG) { g.barrier(); refresh(VEC, ZG); }
  template <int K, int M>
  __device__ void reduce(double (&v)[K + M], double*, int&) { g.template reduce<K, M>(v); }
};

// A resident grid of workgroups (as many as the chip holds at once) works
// through plist[0, count): workgroup b solves item b, then takes the next
// unsolved item from the launch's counter `next` (zero before the launch)
// until none is left.  Pairs are solved in list order (largest first), a
// new pair starts on a workgroup as soon as its previous one ends, and
// every XCD draws from the one queue; each pair's result is independent of
// which workgroup solves it.
template <int T, int VPT>
__global__ void __launch_bounds__(T) k_lm_solve_lds(const LMPairDesc* __restrict__ pairs,
                                                    const int* __restrict__ plist, int count, int* __restrict__ next,
                                                    LMArrays A, LMOptionsDev opt, LMResultDev* __restrict__ res,
                                                    long long totalV, unsigned lds_bytes) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double red[2 * 8 * kMaxWaves];
  __shared__ int scan_buf[kMaxWaves];
  __shared__ int s_item;
  int w = blockIdx.x;
  while (w < count) {
    const int pid = plist[w];
    const LMPairDesc P = pairs[pid];
    LdsSolo team(P.nv);
    lds_solve<T, VPT, LdsSolo, unsigned short>(P, pid, team, A, opt, res, totalV, smem, red, scan_buf, lds_bytes);
    __syncthreads();   // every thread is done with this pair's LDS
    if (threadIdx.x == 0) s_item = (int)gridDim.x + atomicAdd(next, 1);
    __syncthreads();
    w = s_item;
  }
}

// wg[b] = (team, rank, team size, chunk): team t solves pair plist[t];
// workgroup `rank` owns vertices [rank chunk, min(nv, (rank + 1) chunk)).
template <int T, int VPT>
__global__ void __launch_bounds__(T) k_lm_solve_lds_team(const LMPairDesc* __restrict__ pairs,
                                                         const int* __restrict__ plist, const int4* __restrict__ wg,
                                                         LMArrays A, LMOptionsDev opt, LMResultDev* __restrict__ res,
                                                         long long totalV, unsigned* cnt, double* part,
                                                         int* abort_flag, long long limit, unsigned lds_bytes) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double red[2 * 8 * kMaxWaves];
  __shared__ int scan_buf[kMaxWaves];
  const int4 m = wg[blockIdx.x];
  const int pid = plist[m.x];
  const LMPairDesc P = pairs[pid];
  const int lo = min(P.nv, m.y * m.w), hi = min(P.nv, lo + m.w);
  LdsTeam team(CoherentTeam{m.y, m.z, cnt + (size_t)m.x * 32, part + (size_t)m.x * 2 * kMaxTeam * 8, abort_flag, limit,
                            0u, 0},
               lo, hi);
  lds_solve<T, VPT, LdsTeam, unsigned>(P, pid, team, A, opt, res, totalV, smem, red, scan_buf, lds_bytes);
}

__device__ inline unsigned long long* pair_slots(const LMArrays& A, long long totalV, long long vbase) {
  return (unsigned long long*)(A.work + (size_t)gSlots * totalV + vbase);
}

// Large pairs with their halo in LDS; wg as for k_lm_solve_lds_team.  Bound
// by the two exchanges and the halo copy of a PCG iteration (about 10 us at
// three vertices per thread).  1024x3 spills 20 registers, 1024x4 44 (76 and
// 124 bytes of scratch a lane).  Twelve icospheres each of 10242 and 40962
// vertices, 50 steps of 30 PCG iterations: 55.7 ms on k_lm_solve_lds_team,
// whose gather waits for a remote read per neighbour, 14.9 ms here.
template <int T, int VPT>
__global__ void __launch_bounds__(T) k_lm_solve_lds_halo(const LMPairDesc* __restrict__ pairs,
                                                         const int* __restrict__ plist, const int4* __restrict__ wg,
                                                         LMArrays A, LMOptionsDev opt, LMResultDev* __restrict__ res,
                                                         long long totalV, int* abort_flag, long long limit,
                                                         unsigned lds_bytes) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double red[kTagRed];
  __shared__ int scan_buf[kMaxWaves];
  const int4 m = wg[blockIdx.x];
  const int pid = plist[m.x];
  const LMPairDesc P = pairs[pid];
  const int lo = min(P.nv, m.y * m.w), hi = min(P.nv, lo + m.w);
  const int* perm = (const int*)(A.work + (size_t)gOrder * totalV + P.vbase);
  LdsHalo team(TagTeam{m.y, m.z, pair_slots(A, totalV, P.vbase), abort_flag, limit, red, 0u, 0}, lo, hi, perm,
               perm + P.nv);
  lds_solve<T, VPT, LdsHalo, unsigned short>(P, pid, team, A, opt, res, totalV, smem, red, scan_buf, lds_bytes);
}

// Bound on any one wait of a team, in device clock ticks.
int team_wait_limit(long long* limit) {
  int dev = 0, khz = 0;
  MO_HIP(hipGetDevice(&dev));
  MO_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
  *limit = (long long)std::max(khz, 1) * 1000LL * 20;   // 20 s
  if (const char* w = getenv("MO_LM_TEAM_WAIT_US")) *limit = atoll(w) * (long long)std::max(khz, 1) / 1000LL;
  return MO_OK;
}

bool coop_refused_by_host() {
  const char* f = getenv("MO_LM_COOP_REFUSE");
  return f && f[0] == '1';
}

// kCoopRefused when the runtime refuses the cooperative grid (nothing was
// launched then).
int launch_coop(const void* kern, int nwg, int threads, void** args, size_t lds_bytes, hipStream_t s) {
  if (coop_refused_by_host()) return kCoopRefused;
  if (hipLaunchCooperativeKernel(kern, dim3(nwg), dim3(threads), args, (unsigned)lds_bytes, s) != hipSuccess) {
    (void)hipGetLastError();
    return kCoopRefused;
  }
  return MO_OK;
}

int coop_capacity(const void* kern, int threads, size_t lds_bytes) {
  int dev = 0, cus = 0, per = 0;
  if (hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes) != hipSuccess ||
      hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, threads, lds_bytes) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return per * cus;
}

template <int T, int VPT>
int launch_halo_bucket(const LMPairDesc* pairs_dev, const int* plist, const int4* wg_dev, int nwg, const LMArrays& A,
                       const LMOptionsDev& opt, LMResultDev* res, long long totalV, size_t lds_bytes, int* abort_flag,
                       hipStream_t s) {
  auto kern = k_lm_solve_lds_halo<T, VPT>;
  MO_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes));
  long long limit = 0;
  if (int rc = team_wait_limit(&limit)) return rc;
  LMArrays a = A;
  LMOptionsDev o = opt;
  unsigned lb = (unsigned)lds_bytes;
  void* args[] = {(void*)&pairs_dev, (void*)&plist,  (void*)&wg_dev,     (void*)&a,     (void*)&o,
                  (void*)&res,       (void*)&totalV, (void*)&abort_flag, (void*)&limit, (void*)&lb};
  return launch_coop((const void*)kern, nwg, T, args, lds_bytes, s);
}

// Team launch of the register/LDS kernel: nwg workgroups (wg_dev entries)
// in one cooperative grid.
template <int T, int VPT>
int launch_team_bucket(const LMPairDesc* pairs_dev, const int* plist, const int4* wg_dev, int nwg, const LMArrays& A,
                       const LMOptionsDev& opt, LMResultDev* res, long long totalV, size_t lds_bytes, unsigned* cnt,
                       double* part, int* abort_flag, hipStream_t s) {
  auto kern = k_lm_solve_lds_team<T, VPT>;
  MO_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes));
  long long limit = 0;
  if (int rc = team_wait_limit(&limit)) return rc;
  LMArrays a = A;
  LMOptionsDev o = opt;
  long long tv = totalV;
  unsigned lb = (unsigned)lds_bytes;
  void* args[] = {(void*)&pairs_dev, (void*)&plist, (void*)&wg_dev, (void*)&a,           (void*)&o,
                  (void*)&res,       (void*)&tv,    (void*)&cnt,    (void*)&part,        (void*)&abort_flag,
                  (void*)&limit,     (void*)&lb};
  return launch_coop((const void*)kern, nwg, T, args, lds_bytes, s);
}

__host__ __device__ inline size_t lm_lds_bytes_dev(int nv, long long padded_entries) {
  return (((size_t)nv * 16 + 16 + (size_t)padded_entries * 2) + 15) & ~(size_t)15;
}

// Per pair: for each team shape b, the largest chunk's adjacency entries
// (the sum of its vertices' neighbour counts; adjacency rows may have unused
// slots after merging, so row offsets do not give it), then the one-
// workgroup kernel's LDS entries (every vertex's count rounded up to even).
// out[4 p + 0..3].  One workgroup per pair.
__global__ void __launch_bounds__(256) k_chunk_entries(const LMPairDesc* __restrict__ pairs,
                                                       const int2* __restrict__ adj, int np, int c0, int c1, int c2,
                                                       int* __restrict__ out) {
  __shared__ int acc[3][kMaxTeam];
  const int p = blockIdx.x;
  const int nv = pairs[p].nv;
  const long long vb = pairs[p].vbase;
  const int caps[3] = {c0, c1, c2};
  int c[3], ch[3];
  for (int b = 0; b < 3; ++b) {
    c[b] = nv > 0 ? (nv + caps[b] - 1) / caps[b] : 0;
    ch[b] = c[b] > 0 ? (nv + c[b] - 1) / c[b] : 1;
  }
  for (int k = threadIdx.x; k < 3 * kMaxTeam; k += blockDim.x) acc[k / kMaxTeam][k % kMaxTeam] = 0;
  __syncthreads();
  __shared__ int padded;
  if (threadIdx.x == 0) padded = 0;
  int cur[3] = {-1, -1, -1}, sum[3] = {0, 0, 0}, mine = 0;
  for (int i = threadIdx.x; i < nv; i += blockDim.x) {
    const int n = adj[vb + i].y;
    mine += n + (n & 1);
    for (int b = 0; b < 3; ++b) {
      if (c[b] > kMaxTeam) continue;
      const int r = i / ch[b];
      if (r != cur[b]) {
        if (cur[b] >= 0) atomicAdd(&acc[b][cur[b]], sum[b]);
        cur[b] = r;
        sum[b] = 0;
      }
      sum[b] += n;
    }
  }
  for (int b = 0; b < 3; ++b)
    if (cur[b] >= 0) atomicAdd(&acc[b][cur[b]], sum[b]);
  atomicAdd(&padded, mine);
  __syncthreads();
  if (threadIdx.x < 3) {
    const int b = threadIdx.x;
    int mx = 0;
    if (c[b] > kMaxTeam) mx = INT_MAX;   // no team of this shape holds the pair
    else
      for (int r = 0; r < c[b]; ++r) mx = max(mx, acc[b][r]);
    out[4 * p + b] = mx;
  }
  if (threadIdx.x == 3) out[4 * p + 3] = padded;
}

constexpr int kSoloVertices = 8192;   // most vertices of a one-workgroup shape

// Chunks of a halo team: 3072 vertices per workgroup, 4096 beyond
// kMaxTeam of those (0: too large for either).
__host__ __device__ inline int halo_chunk(int nv, int* chunk) {
  for (int cap = 3072; cap <= 4096; cap += 1024) {
    const int c = (nv + cap - 1) / cap;
    if (c > kMaxTeam) continue;
    *chunk = (nv + c - 1) / c;
    return c;
  }
  return 0;
}

// The pairs marked kPairPlan that can't be solved by one register/LDS
// workgroup (lds_cap: its LDS) but by a halo team: the vertices' spatial order (work slot gOrder:
// perm, inv) and minus the team's LDS bytes in out[4 p + 3], which keeps
// the one-workgroup kernel's entry count otherwise.  The order is that of a
// 32^3 grid's Morton codes over the mesh's box, ties by index (a stable
// radix sort).  An icosphere's numbering gives chunks of 2926 vertices up to
// 16154 neighbours elsewhere (every old vertex's are midpoints far behind
// it), this order at most 442; of a 41000-vertex box mesh 416 and 358.  One
// workgroup per pair; runs beside the grid builds (1.1 ms for 24
// icospheres).  They are planned whatever their numbering: also
// where nothing hides it (templates that are there already) it costs no more
// than the halo kernel gives back in the first LM iteration.  Direct kernel
// and halo kernel with its plan, whole calls of one iteration and of a solve:
// 1 pair of 20000 box vertices 2.08 -> 2.09 and 23.2 -> 20.0 ms, 16 of 8200
// 2.24 -> 2.02 and 21.8 -> 17.8, 2 icospheres of 40962 5.02 -> 2.24 and 73.6
// -> 20.5.
constexpr int kPlanThreads = 512;
static_assert(3072 * 2 >= kTagSlotWords, "a pair's team words fit its work slot");
__device__ inline unsigned spread3(unsigned x) {   // bits 0..4 to 0, 3, .. 12
  unsigned r = 0;
  for (int b = 0; b < 5; ++b) r |= (x >> b & 1u) << (3 * b);
  return r;
}
__global__ void __launch_bounds__(kPlanThreads) k_chunk_plan(const LMPairDesc* __restrict__ pairs, LMArrays A,
                                                             long long totalV, int lds_cap, int* __restrict__ out) {
  __shared__ int buf[16 * kPlanThreads];
  __shared__ int scan_buf[kMaxWaves];
  __shared__ double red[2 * 8 * kMaxWaves];
  const int p = blockIdx.x, tid = threadIdx.x;
  const LMPairDesc P = pairs[p];
  const int nv = P.nv;
  int chunk = 0;
  const int c = halo_chunk(nv, &chunk);
  const int padded = out[4 * p + 3];
  if (!(P.flags & kPairPlan) || (nv <= kSoloVertices && padded < 65536 && lm_lds_bytes_dev(nv, padded) <= (size_t)lds_cap)) return;
  unsigned long long* slots = pair_slots(A, totalV, P.vbase);   // the team's words start at zero
  for (int k = tid; k < kTagSlotWords; k += kPlanThreads) slots[k] = 0ull;
  const float4* X0 = A.x0 + P.vbase;
  int* perm = (int*)(A.work + (size_t)gOrder * totalV + P.vbase);
  int* inv = perm + nv;
  int* code = inv + nv;
  int* tmp = code + nv;
  // box, codes
  double box[6];
  for (int k = 0; k < 6; ++k) box[k] = -INFINITY;
  for (int i = tid; i < nv; i += kPlanThreads) {
    const float4 x = X0[i];
    box[0] = fmax(box[0], (double)-x.x); box[1] = fmax(box[1], (double)-x.y); box[2] = fmax(box[2], (double)-x.z);
    box[3] = fmax(box[3], (double)x.x); box[4] = fmax(box[4], (double)x.y); box[5] = fmax(box[5], (double)x.z);
  }
  int sel = 0;
  block_reduce_dpp<0, 6>(box, red, sel);
  const float ext = (float)fmax(fmax(box[3] + box[0], box[4] + box[1]), box[5] + box[2]);
  const float sc = ext > 0.f && ext < INFINITY ? 32.f / ext : 0.f;
  for (int i = tid; i < nv; i += kPlanThreads) {
    const float4 x = X0[i];
    const float f[3] = {(x.x + (float)box[0]) * sc, (x.y + (float)box[1]) * sc, (x.z + (float)box[2]) * sc};
    unsigned m = 0;
    for (int a = 0; a < 3; ++a) m |= spread3((unsigned)fminf(fmaxf(f[a], 0.f), 31.f)) << a;   // NaN: 0
    code[i] = (int)m;
    tmp[i] = i;
  }
  __syncthreads();
  // four passes of a 4-bit radix sort; thread t moves items [t per, (t + 1) per)
  const int per = (nv + kPlanThreads - 1) / kPlanThreads;
  const int i0 = min(nv, tid * per), i1 = min(nv, i0 + per);
  int* src = tmp;
  int* dst = perm;
  for (int pass = 0; pass < 4; ++pass) {
    for (int d = 0; d < 16; ++d) buf[d * kPlanThreads + tid] = 0;
    // (blocks of 8: the loads of a block are in flight together)
    for (int i = i0; i < i1; i += 8) {
      int d[8];
      for (int q = 0; q < 8; ++q) d[q] = code[src[min(i + q, i1 - 1)]];
      for (int q = 0; q < 8; ++q)
        if (i + q < i1) buf[(d[q] >> (4 * pass) & 15) * kPlanThreads + tid]++;
    }
    __syncthreads();
    int sum = 0;
    for (int q = 0; q < 16; ++q) sum += buf[tid * 16 + q];
    int total;
    int at = block_exclusive_scan(sum, scan_buf, total);
    for (int q = 0; q < 16; ++q) {
      const int n = buf[tid * 16 + q];
      buf[tid * 16 + q] = at;
      at += n;
    }
    __syncthreads();
    for (int i = i0; i < i1; i += 8) {
      int v[8], d[8];
      for (int q = 0; q < 8; ++q) v[q] = src[min(i + q, i1 - 1)];
      for (int q = 0; q < 8; ++q) d[q] = code[v[q]];
      for (int q = 0; q < 8; ++q)
        if (i + q < i1) dst[buf[(d[q] >> (4 * pass) & 15) * kPlanThreads + tid]++] = v[q];
    }
    __syncthreads();
    int* t = src;
    src = dst;
    dst = t;
  }
  // four passes: the order is back in tmp
  for (int i = tid; i < nv; i += kPlanThreads) {
    const int v = src[i];
    perm[i] = v;
    inv[v] = i;
  }
  __syncthreads();
  // the largest LDS of the chunks: records and entries
  const int2* ADJ = A.adj + P.vbase;
  const unsigned* NB = A.nbr + P.ebase;
  unsigned* bm = (unsigned*)buf;   // nv <= 32 * 16 * kPlanThreads
  const int nwords = (nv + 31) >> 5;
  int bytes = 0;
  bool ok = true;
  for (int r = 0; r < c; ++r) {
    const int lo = min(nv, r * chunk), own = min(nv, lo + chunk) - lo;
    for (int q = tid; q < nwords; q += kPlanThreads) bm[q] = 0u;
    __syncthreads();
    int ent = 0;
    for (int il = tid; il < own; il += kPlanThreads) {
      const int2 a = ADJ[perm[lo + il]];
      ent += a.y + (a.y & 1);
      for (int e = 0; e < a.y; e += 8) {
        int r8[8];
        for (int q = 0; q < 8; ++q) r8[q] = inv[nb_index(NB[a.x + min(e + q, a.y - 1)])];
        for (int q = 0; q < 8; ++q)
          if ((unsigned)(r8[q] - lo) >= (unsigned)own) atomicOr(&bm[r8[q] >> 5], 1u << (r8[q] & 31));
      }
    }
    __syncthreads();
    int halo = 0;
    for (int q = tid; q < nwords; q += kPlanThreads) halo += __popc(bm[q]);
    int nh, ne;
    block_exclusive_scan(halo, scan_buf, nh);
    block_exclusive_scan(ent, scan_buf, ne);
    const int records = halo_base(own, nv) + nh + 1;
    ok = ok && records <= 32767 && ne <= 65535;
    bytes = max(bytes, records * 16 + (ne + 7) / 8 * 16);
  }
  if (tid == 0 && ok) out[4 * p + 3] = -bytes;
}

template <int T, int VPT>
int launch_bucket(const LMPairDesc* pairs, const int* plist, int count, int max_nv, int* next, const LMArrays& A,
                  const LMOptionsDev& opt, LMResultDev* res, long long totalV, size_t lds_bytes, hipStream_t s) {
  auto kern = k_lm_solve_lds<T, VPT>;
  // one vertex per thread: no more waves than the largest pair needs (idle
  // ones would still take part in every reduction).  One pair's whole call at
  // 32^3 on 16 waves and trimmed: 128 vertices 3.21 -> 2.53 ms, 258 vertices
  // 4.31 -> 3.70, 642 vertices 4.26 -> 4.03, 770 and more the same.
  const int threads = VPT == 1 ? std::min(T, std::max(64, (max_nv + 63) / 64 * 64)) : T;
  MO_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes));
  // one wave of workgroups: the chip's capacity for this shape and LDS size,
  // with the waves of a workgroup counted as a multiple of the CU's four
  // SIMDs.  Ten waves lie 3, 3, 2, 2: a second such workgroup would put a
  // sixth on a SIMD that holds five of this kernel, so it waits for the CU to
  // empty, where a resident workgroup takes the next pair as soon as it has
  // one (280 pairs of 602 vertices, LM: two workgroups counted per CU 9.4 ms,
  // one 7.2; 512 pairs 9.5 either way).
  int dev = 0, cus = 0, per = 0;
  MO_HIP(hipGetDevice(&dev));
  MO_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  MO_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void*)kern, (threads + 255) / 256 * 256,
                                                      lds_bytes));
  const int nwg = std::max(1, std::min(count, std::max(per, 1) * std::max(cus, 1)));
  hipLaunchKernelGGL(kern, dim3(nwg), dim3(threads), lds_bytes, s, pairs, plist, count, next, A, opt, res, totalV,
                     (unsigned)lds_bytes);
  MO_HIP(hipGetLastError());
  return MO_OK;
}

}  // namespace

// Shapes of the register/LDS kernel: (threads, vertices per thread).  A pair
// of nv vertices can use any shape with T * VPT >= nv.  Which one it gets:
//   1. the size-class table, when one is set (lm_lds_set_table: pairs with
//      nv <= max_nv[r], first r in ascending order, use shape[r]; this is
//      what the autotuner installs after timing the candidates);
//   2. else the first fitting shape in the preference order: the built-in
//      order kPref, or MO_LM_SHAPES="TxVPT,TxVPT,..." read once.
static const int kShapeT[] = {1024, 1024, 1024, 1024, 512, 512, 512, 512, 256, 256, 256, 768, 768};
static const int kShapeVPT[] = {1, 2, 4, 5, 8, 10, 12, 16, 20, 24, 32, 6, 7};
constexpr int kNumShapes = 13;
// built-in preference: 768x7 ahead of 1024x5 (5000-vertex pairs: 36.3 against
// 37.3 ms per 512-pair launch; they spill 40 and 46 VGPRs), otherwise by capacity
static const int kPref[kNumShapes] = {0, 1, 2, 12, 3, 4, 11, 5, 6, 7, 8, 9, 10};

static std::mutex g_shape_mu;
static std::vector<int> g_table_nv, g_table_shape;   // guarded by g_shape_mu

static const std::vector<int>& shape_preference() {
  static const std::vector<int> pref = [] {
    std::vector<int> p;
    const char* env = getenv("MO_LM_SHAPES");
    if (env) {
      std::string e(env);
      size_t pos = 0;
      while (pos < e.size()) {
        size_t comma = e.find(',', pos);
        std::string tok = e.substr(pos, comma == std::string::npos ? std::string::npos : comma - pos);
        int t = 0, v = 0;
        if (sscanf(tok.c_str(), "%dx%d", &t, &v) == 2)
          for (int b = 0; b < kNumShapes; ++b)
            if (kShapeT[b] == t && kShapeVPT[b] == v) p.push_back(b);
        if (comma == std::string::npos) break;
        pos = comma + 1;
      }
    }
    if (p.empty()) p.assign(kPref, kPref + kNumShapes);
    return p;
  }();
  return pref;
}

int lm_lds_buckets() { return kNumShapes; }

int lm_lds_shape(int b, int* threads, int* vpt) {
  if (b < 0 || b >= kNumShapes) return fail(MO_ERR_ARG, "shape index %d out of range [0, %d)", b, kNumShapes);
  if (threads) *threads = kShapeT[b];
  if (vpt) *vpt = kShapeVPT[b];
  return MO_OK;
}

int lm_lds_set_table(const int* max_nv, const int* shape, int n) {
  MO_CHECK(n >= 0 && (n == 0 || (max_nv && shape)), MO_ERR_ARG, "shape table: bad arguments");
  for (int r = 0; r < n; ++r) {
    MO_CHECK(shape[r] >= 0 && shape[r] < kNumShapes, MO_ERR_ARG, "shape table row %d: shape %d out of range", r,
             shape[r]);
    MO_CHECK(max_nv[r] >= 1 && (r == 0 || max_nv[r] > max_nv[r - 1]), MO_ERR_ARG,
             "shape table row %d: max_nv must be positive and ascending", r);
    MO_CHECK((long long)kShapeT[shape[r]] * kShapeVPT[shape[r]] >= max_nv[r], MO_ERR_ARG,
             "shape table row %d: shape %dx%d holds fewer than %d vertices", r, kShapeT[shape[r]],
             kShapeVPT[shape[r]], max_nv[r]);
  }
  std::lock_guard<std::mutex> lk(g_shape_mu);
  g_table_nv.assign(max_nv, max_nv + n);
  g_table_shape.assign(shape, shape + n);
  return MO_OK;
}

int lm_lds_bucket_for(int nv) {
  {
    std::lock_guard<std::mutex> lk(g_shape_mu);
    for (size_t r = 0; r < g_table_nv.size(); ++r)
      if (nv <= g_table_nv[r]) return g_table_shape[r];
  }
  for (int b : shape_preference())
    if (nv <= kShapeT[b] * kShapeVPT[b]) return b;
  return -1;
}

// Team shapes of the register/LDS kernel (threads x vertices per thread per
// workgroup), in preference order: the largest chunk whose LDS fits.
static const int kTeamT[] = {1024, 1024, 1024};
static const int kTeamVPT[] = {4, 3, 2};
constexpr int kHaloShape = 3;   // then the halo teams of 1024x3 and 1024x4

int lm_lds_team_shapes() { return kHaloShape + 2; }

// Preference order of the team shapes: 1024x3, then 1024x4 (only for pairs
// whose 3072-vertex team would exceed kMaxTeam), then 1024x2 (chunks whose
// adjacency does not fit the LDS otherwise) -- 1024x3 solved 12k-100k vertex
// pairs as fast as 1024x4 and 4% faster on 41k-vertex icospheres (it spills
// no register, 1024x4 20) -- or
// MO_LM_TEAM_VPT="v,v,..." (vertices per thread, e.g. "2,4") read once.
const std::vector<int>& lm_lds_team_order() {
  static const std::vector<int> order = [] {
    std::vector<int> o;
    if (const char* env = getenv("MO_LM_TEAM_VPT")) {
      std::string e(env);
      size_t pos = 0;
      while (pos <= e.size()) {
        const size_t comma = e.find(',', pos);
        const int v = atoi(e.substr(pos, comma == std::string::npos ? std::string::npos : comma - pos).c_str());
        for (int b = 0; b < 3; ++b)
          if (kTeamVPT[b] == v) o.push_back(b);
        if (comma == std::string::npos) break;
        pos = comma + 1;
      }
    }
    if (o.empty()) o = {1, 0, 2};
    return o;
  }();
  return order;
}

int lm_lds_team_max() { return kMaxTeam; }

int lm_lds_team_shape(int b, int* threads, int* vpt) {
  MO_CHECK(b >= 0 && b < lm_lds_team_shapes(), MO_ERR_ARG, "team shape %d out of range", b);
  *threads = 1024;
  *vpt = b < kHaloShape ? kTeamVPT[b] : 3 + (b - kHaloShape);
  return MO_OK;
}

size_t lm_lds_team_bytes(int chunk, long long entries) {
  return (((size_t)chunk * 16 + (size_t)entries * 4) + 15) & ~(size_t)15;
}

int lm_lds_team_capacity(int b, size_t lds_bytes) {
  switch (b) {
    case 0: return coop_capacity((const void*)k_lm_solve_lds_team<1024, 4>, 1024, lds_bytes);
    case 1: return coop_capacity((const void*)k_lm_solve_lds_team<1024, 3>, 1024, lds_bytes);
    case 2: return coop_capacity((const void*)k_lm_solve_lds_team<1024, 2>, 1024, lds_bytes);
    case kHaloShape: return coop_capacity((const void*)k_lm_solve_lds_halo<1024, 3>, 1024, lds_bytes);
    case kHaloShape + 1: return coop_capacity((const void*)k_lm_solve_lds_halo<1024, 4>, 1024, lds_bytes);
    default: return 0;
  }
}

// A pair is planned where its vertex count, or the adjacency that its edge
// count gives a closed mesh (half the vertices' lists padded by one), is more
// than one workgroup holds.  The counts alone decide, so that a pair's kernel
// does not depend on the batch, and no plan is launched where none is needed:
// its workgroups, two waves per SIMD, do not get in between a running grid
// build's single waves, and for 512 pairs of 5000 vertices, which it leaves
// alone, it held the solver's launch back to that build's end (pipelined
// batches of 512 62.3 ms, without it 60.5; of 256 31.6 and 30.3).  A mesh whose adjacency outgrows the
// estimate takes the direct team kernel.
bool lm_lds_wants_plan(long long nv, long long entries, size_t lds_cap) {
  int chunk = 0;
  const long long padded = entries + nv / 2;
  return nv > 3072 && nv <= (long long)kMaxTeam * 4096 && halo_chunk((int)nv, &chunk) >= 2 &&
         (nv > kSoloVertices || padded >= 65536 || lm_lds_bytes_dev((int)nv, padded) > lds_cap);
}

int lm_lds_chunk_entries(const LMPairDesc* pairs_dev, const LMArrays& A, int np, long long totalV, bool plan,
                         size_t lds_cap, int* out_dev, hipStream_t s) {
  if (np <= 0) return MO_OK;
  hipLaunchKernelGGL(k_chunk_entries, dim3(np), dim3(256), 0, s, pairs_dev, A.adj, np,
                     kTeamT[0] * kTeamVPT[0], kTeamT[1] * kTeamVPT[1], kTeamT[2] * kTeamVPT[2], out_dev);
  MO_HIP(hipGetLastError());
  if (plan) {
    hipLaunchKernelGGL(k_chunk_plan, dim3(np), dim3(kPlanThreads), 0, s, pairs_dev, A, totalV, (int)lds_cap, out_dev);
    MO_HIP(hipGetLastError());
  }
  return MO_OK;
}

int lm_lds_halo_shape(int nv, int* chunk, int* workgroups) {
  *workgroups = halo_chunk(nv, chunk);
  return *workgroups == 0 ? -1 : *chunk <= 3072 ? kHaloShape : kHaloShape + 1;
}

int lm_lds_team_launch(int b, const LMPairDesc* pairs, const int* plist, const int4* wg_dev, int nwg,
                       const LMArrays& A, const LMOptionsDev& opt, LMResultDev* res, long long totalV,
                       size_t lds_bytes, unsigned* cnt, double* part, int* abort_flag, hipStream_t s) {
  if (nwg <= 0) return MO_OK;
  switch (b) {
    case 0: return launch_team_bucket<1024, 4>(pairs, plist, wg_dev, nwg, A, opt, res, totalV, lds_bytes, cnt, part,
                                               abort_flag, s);
    case 1: return launch_team_bucket<1024, 3>(pairs, plist, wg_dev, nwg, A, opt, res, totalV, lds_bytes, cnt, part,
                                               abort_flag, s);
    case 2: return launch_team_bucket<1024, 2>(pairs, plist, wg_dev, nwg, A, opt, res, totalV, lds_bytes, cnt, part,
                                               abort_flag, s);
    case kHaloShape: return launch_halo_bucket<1024, 3>(pairs, plist, wg_dev, nwg, A, opt, res, totalV, lds_bytes,
                                                        abort_flag, s);
    case kHaloShape + 1: return launch_halo_bucket<1024, 4>(pairs, plist, wg_dev, nwg, A, opt, res, totalV, lds_bytes,
                                                            abort_flag, s);
    default: return fail(MO_ERR_ARG, "bad register/LDS team shape %d", b);
  }
}

size_t lm_lds_bytes(int nv, long long padded_entries) {
  return lm_lds_bytes_dev(nv, padded_entries);
}

int lm_lds_launch(int bucket, const LMPairDesc* pairs, const int* plist, int count, int max_nv, int* next, const LMArrays& A,
                  const LMOptionsDev& opt, LMResultDev* res, long long totalV, size_t lds_bytes, hipStream_t s) {
  if (count <= 0) return MO_OK;
  switch (bucket) {
#define MO_SHAPE(ID, T, V) \
    case ID: return launch_bucket<T, V>(pairs, plist, count, max_nv, next, A, opt, res, totalV, lds_bytes, s);
    MO_SHAPE(0, 1024, 1) MO_SHAPE(1, 1024, 2) MO_SHAPE(2, 1024, 4) MO_SHAPE(3, 1024, 5)
    MO_SHAPE(4, 512, 8) MO_SHAPE(5, 512, 10) MO_SHAPE(6, 512, 12) MO_SHAPE(7, 512, 16)
    MO_SHAPE(8, 256, 20) MO_SHAPE(9, 256, 24) MO_SHAPE(10, 256, 32) MO_SHAPE(11, 768, 6) MO_SHAPE(12, 768, 7)
#undef MO_SHAPE
    default: return fail(MO_ERR_ARG, "bad LDS solver shape %d", bucket);
  }
}

}  // namespace mo
