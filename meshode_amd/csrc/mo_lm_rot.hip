// Levenberg-Marquardt solve of Deformer::DeformWithRot (deformer.cc:94-171)
// on gfx950: the whole trust-region loop in one persistent kernel (the loop
// of mo_lm_util.h), on chip on one workgroup per 256-vertex chunk of the
// problem (k_lm_rot_chip below), or, for problems that kernel does not hold
// and where the runtime refuses a cooperative grid, with its vectors in
// global memory, on one workgroup (k_lm_rot) or on a team (k_lm_rot_team).
//
// Unknowns per vertex i: the position p_i = x0_i + u_i and an angle-axis
// rotation w_i (zero at the start, deformer.cc:114).  Residuals:
//   DistanceLoss   d(p_i)                                  (distanceloss.h:6-25)
//   EdgeLossWithRot, per face half-edge h = (a, b) = (F[f][j], F[f][j+1]):
//     lambda (rotate(w_a, p_a - p_b) - v_h),  v_h = x0_a - x0_b,
//     w_a - w_b                                          (edgeloss.h:64-90)
// with the rotation and its derivatives of mo_rotate.h.  The Jacobian of
// half-edge h has the blocks lambda A_a (p_a), -lambda A_a (p_b),
// lambda G_h (w_a) for the first three residuals (A_a = dq/dp at w_a,
// G_h = dq/dw at (w_a, p_a - p_b)) and I (w_a), -I (w_b) for the last three.
//
// Per LM step, (J^T J + D^2) delta = -J^T f is solved by PCG with FP32
// vectors and FP64 reductions; in k_lm_rot J^T J x is formed matrix-free in two passes
// (per half-edge: t = lambda (A_a (x_pa - x_pb) + G_h x_wa) and
// s = x_wa - x_wb and their transposed images; per vertex: the gather over
// its outgoing and incoming half-edges), preconditioned by the inverse of
// each vertex's 6x6 diagonal block of J^T J + D^2.  Jacobi scaling, LM
// diagonal and trust-region decisions are those of the shared loop.
#include <algorithm>
#include <cstdlib>
#include "mo_common.h"
#include "mo_lm.h"
#include "mo_lm_rot.h"
#include "mo_lm_util.h"
#include "mo_lookup.h"
#include "mo_rotate.h"

namespace mo {

namespace {

enum VSlot {
  vG = 0, vA0, vA1, vA2, vSp, vSw, vGRp, vGRw, vDGp, vDGw, vDTp, vDTw,
  vM0, vM1, vM2, vM3, vM4, vM5, vRp, vRw, vZp, vZw, vPp, vPw, vQp, vQw, vDLp, vDLw, vNumSlots
};
enum HSlot { hG0 = 0, hG1, hG2, hSig, hC, hD, hE, hNumSlots };
static_assert(vNumSlots == kRotVSlots && hNumSlots == kRotHSlots, "slot counts are part of the host contract");

__device__ inline float3 f3(const float4 v) { return make_float3(v.x, v.y, v.z); }
__device__ inline float4 f4(const float3 v) { return make_float4(v.x, v.y, v.z, 0.f); }
__device__ inline float3 add(float3 a, float3 b) { return make_float3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ inline float3 sub(float3 a, float3 b) { return make_float3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ inline float3 mul(float3 a, float s) { return make_float3(a.x * s, a.y * s, a.z * s); }
__device__ inline double dot3(float3 a, float3 b) { return (double)a.x * b.x + (double)a.y * b.y + (double)a.z * b.z; }
// M v and M^T v for a matrix stored as three float4 rows
__device__ inline float3 mv(const float4 r0, const float4 r1, const float4 r2, float3 v) {
  return make_float3(r0.x * v.x + r0.y * v.y + r0.z * v.z, r1.x * v.x + r1.y * v.y + r1.z * v.z,
                     r2.x * v.x + r2.y * v.y + r2.z * v.z);
}
__device__ inline float3 mtv(const float4 r0, const float4 r1, const float4 r2, float3 v) {
  return make_float3(r0.x * v.x + r1.x * v.y + r2.x * v.z, r0.y * v.x + r1.y * v.y + r2.y * v.z,
                     r0.z * v.x + r1.z * v.y + r2.z * v.z);
}
__device__ inline float3 absmax3(float3 a) {
  return make_float3(fabsf(a.x), fabsf(a.y), fabsf(a.z));
}

// packed upper triangle of a symmetric 6x6 matrix
__device__ inline int sym6(int r, int c) {
  if (r > c) { const int t = r; r = c; c = t; }
  return r * 6 - (r * (r - 1)) / 2 + (c - r);
}

// Inverse of an SPD 6x6 matrix (FP64 Cholesky); false when not SPD.
__device__ inline bool spd6_inverse(double (&M)[6][6], float (&out)[21]) {
  double L[6][6];
  for (int i = 0; i < 6; ++i)
    for (int j = 0; j <= i; ++j) {
      double s = M[i][j];
      for (int k = 0; k < j; ++k) s -= L[i][k] * L[j][k];
      if (i == j) {
        if (!(s > 0.0)) return false;
        L[i][i] = sqrt(s);
      } else {
        L[i][j] = s / L[j][j];
      }
    }
  // inverse column by column: L L^T x = e_c
  for (int c = 0; c < 6; ++c) {
    double y[6];
    for (int i = 0; i < 6; ++i) {
      double s = (i == c) ? 1.0 : 0.0;
      for (int k = 0; k < i; ++k) s -= L[i][k] * y[k];
      y[i] = s / L[i][i];
    }
    double x[6];
    for (int i = 5; i >= 0; --i) {
      double s = y[i];
      for (int k = i + 1; k < 6; ++k) s -= L[k][i] * x[k];
      x[i] = s / L[i][i];
    }
    for (int r = 0; r <= c; ++r) out[sym6(r, c)] = (float)x[r];
  }
  return true;
}

template <class Team>
__device__ inline void lm_rot_pair(const RotPairDesc P, LMResultDev* out, const RotArrays& A,
                                   const LMOptionsDev& opt, long long totalV, long long totalH, Team& team,
                                   double* red) {
  const int T = blockDim.x, tid = threadIdx.x;
  const int i0 = team.rank() * T + tid, stride = team.size() * T;
  const int nv = P.nv, nh = P.nh;
  const float lam = P.lambda, l2 = lam * lam;
  const float* __restrict__ grid = P.grid;
  const int N = P.N;
  const long long vb = P.vbase, hb = P.hbase;
  const float4* __restrict__ X0 = A.x0 + vb;
  float4* __restrict__ U = A.u + vb;
  float4* __restrict__ WR = A.w + vb;
  const int4* __restrict__ ADJ = A.vadj + vb;
  const int* __restrict__ VL = A.vlist + P.lbase;
  const int2* __restrict__ HAB = A.hab + hb;
  float4* __restrict__ V[vNumSlots];
  for (int k = 0; k < vNumSlots; ++k) V[k] = A.vwork + (size_t)k * totalV + vb;
  float4* __restrict__ H[hNumSlots];
  for (int k = 0; k < hNumSlots; ++k) H[k] = A.hwork + (size_t)k * totalH + hb;
  int sel = 0;
  const long long clock_start = wall_clock64();

  // J^T J diagonal block of vertex i (6x6, p then w), without D^2
  auto vertex_block = [&](int i, double (&M)[6][6]) {
    for (int r = 0; r < 6; ++r)
      for (int c = 0; c < 6; ++c) M[r][c] = 0.0;
    const float4 g = V[vG][i];
    const float gv[3] = {g.x, g.y, g.z};
    for (int r = 0; r < 3; ++r)
      for (int c = 0; c < 3; ++c) M[r][c] += (double)gv[r] * gv[c];
    const int4 adj = ADJ[i];
    const float4 a0 = V[vA0][i], a1 = V[vA1][i], a2 = V[vA2][i];
    const float Ai[9] = {a0.x, a0.y, a0.z, a1.x, a1.y, a1.z, a2.x, a2.y, a2.z};
    // outgoing: l2 A_i^T A_i (p,p), l2 A_i^T G (p,w), l2 G^T G + I (w,w)
    for (int k = 0; k < adj.y; ++k) {
      const int h = VL[adj.x + k];
      const float4 q0 = H[hG0][h], q1 = H[hG1][h], q2 = H[hG2][h];
      const float Gm[9] = {q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, q2.x, q2.y, q2.z};
      for (int r = 0; r < 3; ++r)
        for (int c = 0; c < 3; ++c) {
          double pp = 0, pw = 0, ww = 0;
          for (int m = 0; m < 3; ++m) {
            pp += (double)Ai[3 * m + r] * Ai[3 * m + c];
            pw += (double)Ai[3 * m + r] * Gm[3 * m + c];
            ww += (double)Gm[3 * m + r] * Gm[3 * m + c];
          }
          M[r][c] += l2 * pp;
          M[r][3 + c] += l2 * pw;
          M[3 + c][r] += l2 * pw;
          M[3 + r][3 + c] += l2 * ww + (r == c ? 1.0 : 0.0);
        }
    }
    // incoming: l2 A_a^T A_a (p,p), I (w,w)
    for (int k = 0; k < adj.z; ++k) {
      const int h = VL[adj.x + adj.y + k];
      const int a = HAB[h].x;
      const float4 b0 = V[vA0][a], b1 = V[vA1][a], b2 = V[vA2][a];
      const float Aa[9] = {b0.x, b0.y, b0.z, b1.x, b1.y, b1.z, b2.x, b2.y, b2.z};
      for (int r = 0; r < 3; ++r)
        for (int c = 0; c < 3; ++c) {
          double pp = 0;
          for (int m = 0; m < 3; ++m) pp += (double)Aa[3 * m + r] * Aa[3 * m + c];
          M[r][c] += l2 * pp;
        }
      for (int r = 0; r < 3; ++r) M[3 + r][3 + r] += 1.0;
    }
  };

  auto apply_minv = [&](int i, float3 rp, float3 rw, float3& zp, float3& zw) {
    float m[24];
    for (int k = 0; k < 6; ++k) {
      const float4 t = V[vM0 + k][i];
      m[4 * k] = t.x; m[4 * k + 1] = t.y; m[4 * k + 2] = t.z; m[4 * k + 3] = t.w;
    }
    const float r[6] = {rp.x, rp.y, rp.z, rw.x, rw.y, rw.z};
    float z[6];
    for (int a = 0; a < 6; ++a) {
      float s = 0.f;
      for (int b = 0; b < 6; ++b) s += m[sym6(a, b)] * r[b];
      z[a] = s;
    }
    zp = make_float3(z[0], z[1], z[2]);
    zw = make_float3(z[3], z[4], z[5]);
  };

  // ---- residuals, Jacobian blocks, gradient J^T f, cost -----------------
  auto eval_jacobian = [&](bool first, double& cv, double& ce, double& gmax) {
    double v[3] = {0.0, 0.0, 0.0};
    for (int i = i0; i < nv; i += stride) {
      const float4 x0 = X0[i], ui = U[i], wi = WR[i];
      const JetF J = lookup_jet(grid, N, x0.x + ui.x, x0.y + ui.y, x0.z + ui.z);
      V[vG][i] = make_float4(J.v0, J.v1, J.v2, J.a);
      const float w[3] = {wi.x, wi.y, wi.z};
      float Am[9];
      rotation_point_jacobian(w, Am);
      V[vA0][i] = make_float4(Am[0], Am[1], Am[2], 0.f);
      V[vA1][i] = make_float4(Am[3], Am[4], Am[5], 0.f);
      V[vA2][i] = make_float4(Am[6], Am[7], Am[8], 0.f);
      v[0] += 0.5 * (double)J.a * (double)J.a;
    }
    team.barrier();
    for (int h = i0; h < nh; h += stride) {
      const int2 ab = HAB[h];
      const float4 xa = X0[ab.x], xb = X0[ab.y], ua = U[ab.x], ub = U[ab.y], wa = WR[ab.x], wb = WR[ab.y];
      const float3 vh = make_float3(xa.x - xb.x, xa.y - xb.y, xa.z - xb.z);
      const float e[3] = {vh.x + (ua.x - ub.x), vh.y + (ua.y - ub.y), vh.z + (ua.z - ub.z)};
      const float w[3] = {wa.x, wa.y, wa.z};
      float q[3], G[9];
      rotate_point_dw(w, e, q, G);
      const float3 r = make_float3(lam * (q[0] - vh.x), lam * (q[1] - vh.y), lam * (q[2] - vh.z));
      const float3 sg = make_float3(wa.x - wb.x, wa.y - wb.y, wa.z - wb.z);
      const float4 g0 = make_float4(G[0], G[1], G[2], r.x), g1 = make_float4(G[3], G[4], G[5], r.y),
                   g2 = make_float4(G[6], G[7], G[8], r.z);
      H[hG0][h] = g0;
      H[hG1][h] = g1;
      H[hG2][h] = g2;
      H[hSig][h] = f4(sg);
      const float3 c = mul(mtv(V[vA0][ab.x], V[vA1][ab.x], V[vA2][ab.x], r), lam);
      const float3 d = add(mul(mtv(g0, g1, g2, r), lam), sg);
      H[hC][h] = f4(c);
      H[hD][h] = f4(d);
      v[1] += 0.5 * (dot3(r, r) + dot3(sg, sg));
    }
    team.barrier();
    for (int i = i0; i < nv; i += stride) {
      const float4 g = V[vG][i];
      const int4 adj = ADJ[i];
      float3 gp = make_float3(g.w * g.x, g.w * g.y, g.w * g.z), gw = make_float3(0.f, 0.f, 0.f);
      for (int k = 0; k < adj.y; ++k) {
        const int h = VL[adj.x + k];
        gp = add(gp, f3(H[hC][h]));
        gw = add(gw, f3(H[hD][h]));
      }
      for (int k = 0; k < adj.z; ++k) {
        const int h = VL[adj.x + adj.y + k];
        gp = sub(gp, f3(H[hC][h]));
        gw = sub(gw, f3(H[hSig][h]));
      }
      V[vGRp][i] = f4(gp);
      V[vGRw][i] = f4(gw);
      const float3 m1 = absmax3(gp), m2 = absmax3(gw);
      const float gm = fmaxf(fmaxf(fmaxf(m1.x, m1.y), fmaxf(m1.z, m2.x)), fmaxf(m2.y, m2.z));
      v[2] = (double)gm > v[2] ? (double)gm : v[2];
      if (first) {
        double M[6][6];
        vertex_block(i, M);
        float s[6];
        for (int k = 0; k < 6; ++k) s[k] = (float)(1.0 / (1.0 + sqrt(M[k][k])));
        V[vSp][i] = make_float4(s[0], s[1], s[2], 0.f);
        V[vSw][i] = make_float4(s[3], s[4], s[5], 0.f);
      }
    }
    team.template reduce<2, 1>(v, red, sel);
    cv = v[0]; ce = v[1]; gmax = v[2];
  };

  // ---- LM diagonal, 6x6 block preconditioner, PCG start ----------------
  auto setup_linear = [&](bool reuse, double radius, double& rz_out, double& rr_out) {
    double v[2] = {0.0, 0.0};
    const double inv_radius = 1.0 / radius;
    for (int i = i0; i < nv; i += stride) {
      double M[6][6];
      vertex_block(i, M);
      const float4 sp = V[vSp][i], sw = V[vSw][i];
      const float s[6] = {sp.x, sp.y, sp.z, sw.x, sw.y, sw.z};
      float dg[6];
      if (!reuse) {
        for (int k = 0; k < 6; ++k) {
          double t = (double)s[k] * s[k] * M[k][k];
          t = t < opt.min_lm_diagonal ? opt.min_lm_diagonal : (t > opt.max_lm_diagonal ? opt.max_lm_diagonal : t);
          dg[k] = (float)t;
        }
        V[vDGp][i] = make_float4(dg[0], dg[1], dg[2], 0.f);
        V[vDGw][i] = make_float4(dg[3], dg[4], dg[5], 0.f);
      } else {
        const float4 a = V[vDGp][i], b = V[vDGw][i];
        dg[0] = a.x; dg[1] = a.y; dg[2] = a.z; dg[3] = b.x; dg[4] = b.y; dg[5] = b.z;
      }
      float dt[6];
      for (int k = 0; k < 6; ++k) {
        const double t = (double)dg[k] / ((double)s[k] * s[k]) * inv_radius;
        dt[k] = (float)(t < 1e30 ? t : 1e30);
        M[k][k] += dt[k];
      }
      V[vDTp][i] = make_float4(dt[0], dt[1], dt[2], 0.f);
      V[vDTw][i] = make_float4(dt[3], dt[4], dt[5], 0.f);
      float inv[21];
      if (!spd6_inverse(M, inv)) {
        for (int k = 0; k < 21; ++k) inv[k] = 0.f;
        for (int k = 0; k < 6; ++k) inv[sym6(k, k)] = M[k][k] > 0.0 ? (float)(1.0 / M[k][k]) : 0.f;
      }
      for (int k = 0; k < 5; ++k)
        V[vM0 + k][i] = make_float4(inv[4 * k], inv[4 * k + 1], inv[4 * k + 2], inv[4 * k + 3]);
      V[vM5][i] = make_float4(inv[20], 0.f, 0.f, 0.f);
      const float3 rp = mul(f3(V[vGRp][i]), -1.f), rw = mul(f3(V[vGRw][i]), -1.f);
      float3 zp, zw;
      apply_minv(i, rp, rw, zp, zw);
      V[vRp][i] = f4(rp);
      V[vRw][i] = f4(rw);
      V[vZp][i] = f4(zp);
      V[vZw][i] = f4(zw);
      V[vPp][i] = f4(zp);
      V[vPw][i] = f4(zw);
      V[vDLp][i] = make_float4(0.f, 0.f, 0.f, 0.f);
      V[vDLw][i] = make_float4(0.f, 0.f, 0.f, 0.f);
      v[0] += dot3(rp, zp) + dot3(rw, zw);
      v[1] += dot3(rp, rp) + dot3(rw, rw);
    }
    team.template reduce<2, 0>(v, red, sel);
    rz_out = v[0];
    rr_out = v[1];
  };

  // ---- matrix-free PCG ---------------------------------------------------
  auto pcg = [&](double rz, double rr0) -> int {
    const double tol2 = (double)opt.pcg_relative_tolerance * opt.pcg_relative_tolerance * rr0;
    if (!(rr0 > 0.0)) return 0;
    int k = 0;
    for (; k < opt.pcg_max_iterations; ++k) {
      for (int h = i0; h < nh; h += stride) {
        const int2 ab = HAB[h];
        const float3 pa = f3(V[vPp][ab.x]), pb = f3(V[vPp][ab.y]);
        const float3 wa = f3(V[vPw][ab.x]), wb = f3(V[vPw][ab.y]);
        const float4 a0 = V[vA0][ab.x], a1 = V[vA1][ab.x], a2 = V[vA2][ab.x];
        const float4 g0 = H[hG0][h], g1 = H[hG1][h], g2 = H[hG2][h];
        const float3 t = mul(add(mv(a0, a1, a2, sub(pa, pb)), mv(g0, g1, g2, wa)), lam);
        const float3 s = sub(wa, wb);
        H[hC][h] = f4(mul(mtv(a0, a1, a2, t), lam));
        H[hD][h] = f4(add(mul(mtv(g0, g1, g2, t), lam), s));
        H[hE][h] = f4(s);
      }
      team.barrier();
      double v1[1] = {0.0};
      for (int i = i0; i < nv; i += stride) {
        const float3 pp = f3(V[vPp][i]), pw = f3(V[vPw][i]);
        const float4 g = V[vG][i];
        const float gd = g.x * pp.x + g.y * pp.y + g.z * pp.z;
        const float4 dtp = V[vDTp][i], dtw = V[vDTw][i];
        float3 qp = make_float3(g.x * gd + dtp.x * pp.x, g.y * gd + dtp.y * pp.y, g.z * gd + dtp.z * pp.z);
        float3 qw = make_float3(dtw.x * pw.x, dtw.y * pw.y, dtw.z * pw.z);
        const int4 adj = ADJ[i];
        for (int e = 0; e < adj.y; ++e) {
          const int h = VL[adj.x + e];
          qp = add(qp, f3(H[hC][h]));
          qw = add(qw, f3(H[hD][h]));
        }
        for (int e = 0; e < adj.z; ++e) {
          const int h = VL[adj.x + adj.y + e];
          qp = sub(qp, f3(H[hC][h]));
          qw = sub(qw, f3(H[hE][h]));
        }
        V[vQp][i] = f4(qp);
        V[vQw][i] = f4(qw);
        v1[0] += dot3(pp, qp) + dot3(pw, qw);
      }
      team.template reduce<1, 0>(v1, red, sel);
      const double pq = v1[0];
      if (!(pq > 0.0)) break;
      const float fa = (float)(rz / pq);
      double v2[2] = {0.0, 0.0};
      for (int i = i0; i < nv; i += stride) {
        const float3 pp = f3(V[vPp][i]), pw = f3(V[vPw][i]);
        V[vDLp][i] = f4(add(f3(V[vDLp][i]), mul(pp, fa)));
        V[vDLw][i] = f4(add(f3(V[vDLw][i]), mul(pw, fa)));
        const float3 rp = sub(f3(V[vRp][i]), mul(f3(V[vQp][i]), fa));
        const float3 rw = sub(f3(V[vRw][i]), mul(f3(V[vQw][i]), fa));
        V[vRp][i] = f4(rp);
        V[vRw][i] = f4(rw);
        float3 zp, zw;
        apply_minv(i, rp, rw, zp, zw);
        V[vZp][i] = f4(zp);
        V[vZw][i] = f4(zw);
        v2[0] += dot3(rp, zp) + dot3(rw, zw);
        v2[1] += dot3(rp, rp) + dot3(rw, rw);
      }
      team.template reduce<2, 0>(v2, red, sel);
      const float fb = (float)(v2[0] / rz);
      rz = v2[0];
      if (v2[1] <= tol2) { ++k; break; }
      for (int i = i0; i < nv; i += stride) {
        V[vPp][i] = f4(add(f3(V[vZp][i]), mul(f3(V[vPp][i]), fb)));
        V[vPw][i] = f4(add(f3(V[vZw][i]), mul(f3(V[vPw][i]), fb)));
      }
      team.barrier();
    }
    return k;
  };

  // ---- model cost change, candidate cost, step and parameter norms ------
  auto eval_candidate = [&]() -> LMCandidate {
    double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int i = i0; i < nv; i += stride) {
      const float4 x0 = X0[i], ui = U[i], wi = WR[i];
      const float3 dp = f3(V[vDLp][i]), dw = f3(V[vDLw][i]);
      const float4 g = V[vG][i];
      const float gd = g.x * dp.x + g.y * dp.y + g.z * dp.z;
      v[0] += (double)gd * ((double)g.w + 0.5 * (double)gd);
      const float dc = lookup_f32(grid, N, x0.x + (ui.x + dp.x), x0.y + (ui.y + dp.y), x0.z + (ui.z + dp.z));
      v[1] += 0.5 * (double)dc * (double)dc;
      v[3] += dot3(dp, dp) + dot3(dw, dw);
      const float3 x = make_float3(x0.x + ui.x, x0.y + ui.y, x0.z + ui.z);
      v[4] += dot3(x, x) + dot3(f3(wi), f3(wi));
    }
    for (int h = i0; h < nh; h += stride) {
      const int2 ab = HAB[h];
      const float3 dpa = f3(V[vDLp][ab.x]), dpb = f3(V[vDLp][ab.y]);
      const float3 dwa = f3(V[vDLw][ab.x]), dwb = f3(V[vDLw][ab.y]);
      const float4 a0 = V[vA0][ab.x], a1 = V[vA1][ab.x], a2 = V[vA2][ab.x];
      const float4 g0 = H[hG0][h], g1 = H[hG1][h], g2 = H[hG2][h];
      const float3 r = make_float3(g0.w, g1.w, g2.w), sg = f3(H[hSig][h]);
      const float3 m = mul(add(mv(a0, a1, a2, sub(dpa, dpb)), mv(g0, g1, g2, dwa)), lam);
      const float3 ms = sub(dwa, dwb);
      v[0] += dot3(m, make_float3(r.x + 0.5f * m.x, r.y + 0.5f * m.y, r.z + 0.5f * m.z)) +
              dot3(ms, make_float3(sg.x + 0.5f * ms.x, sg.y + 0.5f * ms.y, sg.z + 0.5f * ms.z));
      const float4 xa = X0[ab.x], xb = X0[ab.y], ua = U[ab.x], ub = U[ab.y], wa = WR[ab.x], wb = WR[ab.y];
      const float3 vh = make_float3(xa.x - xb.x, xa.y - xb.y, xa.z - xb.z);
      const float e[3] = {vh.x + ((ua.x + dpa.x) - (ub.x + dpb.x)), vh.y + ((ua.y + dpa.y) - (ub.y + dpb.y)),
                          vh.z + ((ua.z + dpa.z) - (ub.z + dpb.z))};
      const float w[3] = {wa.x + dwa.x, wa.y + dwa.y, wa.z + dwa.z};
      float q[3];
      rotate_point(w, e, q);
      const float3 rc = make_float3(lam * (q[0] - vh.x), lam * (q[1] - vh.y), lam * (q[2] - vh.z));
      const float3 sc = make_float3(w[0] - (wb.x + dwb.x), w[1] - (wb.y + dwb.y), w[2] - (wb.z + dwb.z));
      v[2] += 0.5 * (dot3(rc, rc) + dot3(sc, sc));
    }
    team.template reduce<5, 0>(v, red, sel);
    return LMCandidate{-v[0], v[1] + v[2], sqrt(v[3]), sqrt(v[4])};
  };

  auto eval = [&](bool first, double& cv, double& ce, double& gmax) { eval_jacobian(first, cv, ce, gmax); };
  auto solve = [&](bool reuse, double radius) -> int {
    double rz, rr;
    setup_linear(reuse, radius, rz, rr);
    return pcg(rz, rr);
  };
  auto accept = [&]() {
    for (int i = i0; i < nv; i += stride) {
      U[i] = f4(add(f3(U[i]), f3(V[vDLp][i])));
      WR[i] = f4(add(f3(WR[i]), f3(V[vDLw][i])));
    }
    team.barrier();
  };
  lm_trust_region_loop(opt, eval, solve, eval_candidate, accept, team.leader() ? out : nullptr, clock_start);
}

__global__ void __launch_bounds__(256) k_lm_rot(const RotPairDesc* __restrict__ pairs, RotArrays A,
                                                 LMOptionsDev opt, LMResultDev* __restrict__ res, long long totalV,
                                                 long long totalH) {
  __shared__ double red[2 * 8 * kMaxWaves];
  const int pid = blockIdx.x;
  SoloTeam team;
  lm_rot_pair(pairs[pid], res + pid, A, opt, totalV, totalH, team, red);
}

// The same on a team of workgroups, for problems the on-chip solver below
// does not hold when the caller asks for teams (options.team_vertices).
// 33024 vertices, 5 steps of 40 PCG iterations: 343 ms on one workgroup of
// 256 threads, 18.2 on 32 of them (46.4 on 32 of 64 threads, 1131 on one).
// wg[b] = (team, rank, team size, -): team t solves problem plist[t].
__global__ void __launch_bounds__(256) k_lm_rot_team(const RotPairDesc* __restrict__ pairs,
                                                      const int* __restrict__ plist, const int4* __restrict__ wg,
                                                      RotArrays A, LMOptionsDev opt, LMResultDev* __restrict__ res,
                                                      long long totalV, long long totalH, unsigned* cnt, double* part,
                                                      int* abort_flag, long long limit) {
  __shared__ double red[2 * 8 * kMaxWaves];
  const int4 m = wg[blockIdx.x];
  const int pid = plist[m.x];
  GridTeam team{m.y, m.z, cnt + (size_t)m.x * 32, part + (size_t)m.x * 2 * kMaxTeam * 8, abort_flag, limit, 0u, 0};
  lm_rot_pair(pairs[pid], res + pid, A, opt, totalV, totalH, team, red);
}

// ---------------------------------------------------------------------------
// The on-chip solver.  With R = A_a (a rotation: A^T A = I) and J = the right
// Jacobian of the exponential map at w_a, dq/dw x = R ((J x) x e), so for a
// half-edge h = (a, b) with e = p_a - p_b the residual's directional
// derivative is
//     lambda R y,   y = x_pa - x_pb + omega_a x e,   omega_a = J x_wa,
// and its transpose images are lambda^2 y at p_a, -lambda^2 y at p_b and
// lambda^2 J^T (e x y) at w_a: no matrix per half-edge is left, and a vertex
// needs nine floats of each neighbour (x_p, x_w, omega) and the edge vector.
// (In the first-order branch, |w|^2 <= double epsilon, J = I and A = I + [w]x
// is orthogonal to 1e-16.)
//
// One thread per vertex holds the vertex's whole PCG state in registers; a
// workgroup holds a chunk of consecutive vertices, its LDS the chunk's
// records and its halo's, and the adjacency with the edge vectors.  A PCG
// iteration publishes z = M^-1 r once, loads the halo's records, forms
// A z, p = z + beta p and A p = A z + beta A p_prev, and needs the two
// reductions of CG and no other exchange; the team protocol is TagTeam.  (A p
// is thus a recurrence, where k_lm_rot forms each product anew.  Whole solves
// of ten box unions of 300 to 5000 vertices, 2 to 6 thousand PCG iterations,
// here and there: the same number of PCG iterations within 3%, final costs
// -3e-6 to 4e-5 apart.)
// What bounds it: the two exchanges and the halo load of an iteration, each
// a round trip through memory shared by the XCDs, not arithmetic (about
// 5.7 us an iteration).  One 5000-vertex problem (20 chunks, 4600 PCG
// iterations): 26.3 ms, where k_lm_rot takes 990 ms on its one CU.  Chunks
// of 256 put one wavefront on each SIMD of a CU; both instances spill 21 VGPRs
// (84 bytes a lane).
__device__ inline float3 cross3(float3 a, float3 b) {
  return make_float3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
__device__ inline float dotf(float3 a, float3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ inline float3 madd(float3 a, float s, float3 b) {   // a + s b
  return make_float3(a.x + s * b.x, a.y + s * b.y, a.z + s * b.z);
}
__device__ inline float3 m9v(const float (&m)[9], float3 v) {
  return make_float3(m[0] * v.x + m[1] * v.y + m[2] * v.z, m[3] * v.x + m[4] * v.y + m[5] * v.z,
                     m[6] * v.x + m[7] * v.y + m[8] * v.z);
}
__device__ inline float3 m9tv(const float (&m)[9], float3 v) {
  return make_float3(m[0] * v.x + m[3] * v.y + m[6] * v.z, m[1] * v.x + m[4] * v.y + m[7] * v.z,
                     m[2] * v.x + m[5] * v.y + m[8] * v.z);
}

// Right Jacobian of the rotation at w: I - a [w]x + b [w]x^2 with
// a = (1 - cos t) / t^2 = 2 sin^2(t / 2) / t^2, b = (t - sin t) / t^3 (its
// series below t = 1, where the difference cancels); I in the first-order
// branch.
__device__ inline void right_jacobian(const float3 w, float (&J)[9]) {
  const float t2 = dotf(w, w);
  float a = 0.f, b = 0.f;
  if (t2 > kAngleAxisEps) {
    const float t = sqrtf(t2);
    const float h = sinf(0.5f * t);
    a = 2.f * h * h / t2;
    b = t2 < 1.f ? 1.f / 6.f + t2 * (-1.f / 120.f + t2 * (1.f / 5040.f + t2 * (-1.f / 362880.f + t2 / 39916800.f)))
                 : (t - sinf(t)) / (t2 * t);
  }
  const float d = 1.f - b * t2;
  J[0] = d + b * w.x * w.x;     J[1] = b * w.x * w.y + a * w.z; J[2] = b * w.x * w.z - a * w.y;
  J[3] = b * w.x * w.y - a * w.z; J[4] = d + b * w.y * w.y;     J[5] = b * w.y * w.z + a * w.x;
  J[6] = b * w.x * w.z + a * w.y; J[7] = b * w.y * w.z - a * w.x; J[8] = d + b * w.z * w.z;
}

__device__ inline unsigned long long pack2(float a, float b) {
  return (unsigned long long)__float_as_uint(a) | ((unsigned long long)__float_as_uint(b) << 32);
}

template <int T>
__global__ void __launch_bounds__(T, T == 256 ? 2 : 1) k_lm_rot_chip(
    const RotPairDesc* __restrict__ pairs, const RotChunk* __restrict__ chunks, RotChipArrays A, LMOptionsDev opt,
    LMResultDev* __restrict__ res, unsigned long long* slots, int* abort_flag, long long limit) {
  extern __shared__ __align__(16) float4 smem4[];
  __shared__ double red[kTagRed];
  const RotChunk C = chunks[blockIdx.x];
  const RotPairDesc P = pairs[C.pid];
  float4* __restrict__ REC = smem4;                                // 3 float4 per record
  float4* __restrict__ LE = smem4 + 3 * (T + C.nhalo);             // edge vector and packed entry
  const int tid = threadIdx.x;
  const bool mine = tid < C.own;
  const int i = C.lo + (mine ? tid : 0);
  const long long vi = P.vbase + i;
  const float lam = P.lambda, l2 = lam * lam;
  TagTeam team{C.rank, C.size, slots + (size_t)C.team * kTagSlotWords, abort_flag, limit, red, 0u, 0};
  const long long clock_start = wall_clock64();
  const int2 row = A.row[vi];
  const int e0 = mine ? row.x : 0, e1 = mine ? row.x + row.y : 0;
  const unsigned* __restrict__ ENT = A.ent + C.ent;
  float4* __restrict__ EV = A.ev + C.ent;
  float4* __restrict__ ER = A.er + C.ent;
  float4* __restrict__ ES = A.es + C.ent;
  const int* __restrict__ HALO = A.halo + C.halo;
  unsigned long long* PUB = A.pub + P.vbase * kRotPubWords;

  const float3 x0 = f3(A.x0[vi]);
  float3 u = f3(A.u[vi]), w = f3(A.w[vi]);
  float3 g = make_float3(0.f, 0.f, 0.f), gp = g, gw = g;
  float dist = 0.f;
  float J[9];                       // right Jacobian at w
  double S1[3], S2[6];              // sums over outgoing edges: e, |e|^2 I - e e^T
  float cnt = 0.f;                  // half-edges at the vertex
  float sc[6], dg[6], dt[6], Mi[21];
  float3 zp, zw, zo, pp, pw, qp, qw, rp, rw, dlp, dlw;
  dlp = dlw = pp = pw = qp = qw = rp = rw = zp = zw = zo = make_float3(0.f, 0.f, 0.f);
  for (int k = 0; k < 6; ++k) sc[k] = dg[k] = dt[k] = 0.f;

  // this vertex's nine published floats, to LDS and, for teams, to memory
  auto publish = [&](float3 a, float3 b, float3 c) {
    if (!mine) return;
    REC[3 * tid] = make_float4(a.x, a.y, a.z, b.x);
    REC[3 * tid + 1] = make_float4(b.y, b.z, c.x, c.y);
    REC[3 * tid + 2].x = c.z;
    if (C.size > 1) {
      unsigned long long* d = PUB + (size_t)i * kRotPubWords;
      const unsigned long long v[kRotPubWords] = {pack2(a.x, a.y), pack2(a.z, b.x), pack2(b.y, b.z), pack2(c.x, c.y),
                                                  pack2(c.z, 0.f)};
      for (int k = 0; k < kRotPubWords; ++k)
        __hip_atomic_store(d + k, v[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  };
  // the halo's records, after the exchange that ended their publication
  auto stage = [&]() {
    for (int k = tid; k < C.nhalo; k += T) {
      unsigned long long* d = PUB + (size_t)HALO[k] * kRotPubWords;
      unsigned long long v[kRotPubWords];
      for (int q = 0; q < kRotPubWords; ++q) v[q] = __hip_atomic_load(d + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      float f[2 * kRotPubWords];
      for (int q = 0; q < kRotPubWords; ++q) {
        f[2 * q] = __uint_as_float((unsigned)v[q]);
        f[2 * q + 1] = __uint_as_float((unsigned)(v[q] >> 32));
      }
      float4* R = REC + 3 * (T + k);
      R[0] = make_float4(f[0], f[1], f[2], f[3]);
      R[1] = make_float4(f[4], f[5], f[6], f[7]);
      R[2].x = f[8];
    }
    if (C.nhalo) __syncthreads();
  };
  auto record = [&](unsigned e, float3& a, float3& b, float3& c) {
    const float4* R = REC + 3 * (e & 0xFFFFFu);
    const float4 r0 = R[0], r1 = R[1];
    a = make_float3(r0.x, r0.y, r0.z);
    b = make_float3(r0.w, r1.x, r1.y);
    c = make_float3(r1.z, r1.w, R[2].x);
  };
  auto out_mult = [](unsigned e) { return (float)((e >> 20) & 63u); };
  auto in_mult = [](unsigned e) { return (float)(e >> 26); };

  // ---- residuals, gradient J^T f, edge vectors and block sums, cost --------
  auto eval = [&](bool first, double& cv, double& ce, double& gmax) {
    publish(u, w, x0);
    team.barrier();
    stage();
    double v[3] = {0.0, 0.0, 0.0};
    if (mine) {
      const JetF L = lookup_jet(P.grid, P.N, x0.x + u.x, x0.y + u.y, x0.z + u.z);
      g = make_float3(L.v0, L.v1, L.v2);
      dist = L.a;
      v[0] = 0.5 * (double)dist * (double)dist;
      const float wv[3] = {w.x, w.y, w.z};
      float Am[9];
      rotation_point_jacobian(wv, Am);
      right_jacobian(w, J);
      gp = mul(g, dist);
      gw = make_float3(0.f, 0.f, 0.f);
      float3 tor = gw;
      cnt = 0.f;
      for (int k = 0; k < 3; ++k) S1[k] = 0.0;
      for (int k = 0; k < 6; ++k) S2[k] = 0.0;
      for (int k = e0; k < e1; ++k) {
        const unsigned pk = ENT[k];
        float3 un, wn, xn;
        record(pk, un, wn, xn);
        const float mo = out_mult(pk), mi = in_mult(pk);
        const float3 vh = sub(x0, xn);
        const float3 e = add(vh, sub(u, un));
        const float3 sg = sub(w, wn);
        LE[k] = make_float4(e.x, e.y, e.z, __uint_as_float(pk));
        float3 cr = make_float3(0.f, 0.f, 0.f);
        if (mo > 0.f) {
          const float3 r = mul(sub(m9v(Am, e), vh), lam);
          const float3 t = mul(m9tv(Am, r), lam);
          cr = t;
          gp = madd(gp, mo, t);
          tor = madd(tor, mo, cross3(e, t));
          v[1] += 0.5 * (double)mo * (dot3(r, r) + dot3(sg, sg));
          const double ex = e.x, ey = e.y, ez = e.z, m = mo;
          S1[0] += m * ex; S1[1] += m * ey; S1[2] += m * ez;
          S2[0] += m * (ey * ey + ez * ez); S2[1] -= m * ex * ey; S2[2] -= m * ex * ez;
          S2[3] += m * (ex * ex + ez * ez); S2[4] -= m * ey * ez; S2[5] += m * (ex * ex + ey * ey);
        }
        if (mi > 0.f) {          // half-edge (j, i): its edge vector is -e, its rest edge -vh
          const float wj[3] = {wn.x, wn.y, wn.z};
          float Aj[9];
          rotation_point_jacobian(wj, Aj);
          const float3 r = mul(sub(vh, m9v(Aj, e)), lam);
          gp = madd(gp, -mi * lam, m9tv(Aj, r));
        }
        gw = madd(gw, mo + mi, sg);
        cnt += mo + mi;
        EV[k] = f4(vh);
        ER[k] = f4(cr);
        ES[k] = f4(sg);
      }
      gw = add(gw, m9tv(J, tor));
      const float3 m1 = absmax3(gp), m2 = absmax3(gw);
      v[2] = (double)fmaxf(fmaxf(fmaxf(m1.x, m1.y), fmaxf(m1.z, m2.x)), fmaxf(m2.y, m2.z));
    }
    team.template reduce<2, 1>(v);
    cv = v[0]; ce = v[1]; gmax = v[2];
    (void)first;
  };

  // J^T J diagonal block (6x6, p then w): g g^T + l2 cnt I, -l2 [S1]x J, l2 J^T S2 J + cnt I
  auto block = [&](double (&M)[6][6]) {
    const double gv[3] = {g.x, g.y, g.z};
    const double K1[3][3] = {{0.0, -S1[2], S1[1]}, {S1[2], 0.0, -S1[0]}, {-S1[1], S1[0], 0.0}};
    const double K2[3][3] = {{S2[0], S2[1], S2[2]}, {S2[1], S2[3], S2[4]}, {S2[2], S2[4], S2[5]}};
    for (int r = 0; r < 3; ++r)
      for (int c = 0; c < 3; ++c) {
        M[r][c] = gv[r] * gv[c] + (r == c ? (double)l2 * cnt : 0.0);
        double pwv = 0.0, wwv = 0.0;
        for (int m = 0; m < 3; ++m) {
          pwv -= K1[r][m] * (double)J[3 * m + c];
          double t = 0.0;
          for (int q = 0; q < 3; ++q) t += K2[m][q] * (double)J[3 * q + c];
          wwv += (double)J[3 * m + r] * t;
        }
        M[r][3 + c] = l2 * pwv;
        M[3 + c][r] = l2 * pwv;
        M[3 + r][3 + c] = l2 * wwv + (r == c ? (double)cnt : 0.0);
      }
  };
  auto minv = [&](float3 a, float3 b, float3& ya, float3& yb) {
    const float r[6] = {a.x, a.y, a.z, b.x, b.y, b.z};
    float y[6];
#pragma unroll
    for (int m = 0; m < 6; ++m) {
      float t = 0.f;
#pragma unroll
      for (int n = 0; n < 6; ++n) t += Mi[sym6(m, n)] * r[n];
      y[m] = t;
    }
    ya = make_float3(y[0], y[1], y[2]);
    yb = make_float3(y[3], y[4], y[5]);
  };

  bool scaled = false;
  // ---- LM diagonal, preconditioner, PCG ------------------------------------
  auto solve = [&](bool reuse, double radius) -> int {
    double v[2] = {0.0, 0.0};
    if (mine) {
      const double inv_radius = 1.0 / radius;
      double M[6][6];
      block(M);
      if (!scaled)
        for (int k = 0; k < 6; ++k) sc[k] = (float)(1.0 / (1.0 + sqrt(M[k][k])));
      if (!reuse)
        for (int k = 0; k < 6; ++k) {
          double t = (double)sc[k] * sc[k] * M[k][k];
          t = t < opt.min_lm_diagonal ? opt.min_lm_diagonal : (t > opt.max_lm_diagonal ? opt.max_lm_diagonal : t);
          dg[k] = (float)t;
        }
      for (int k = 0; k < 6; ++k) {
        const double t = (double)dg[k] / ((double)sc[k] * sc[k]) * inv_radius;
        dt[k] = (float)(t < 1e30 ? t : 1e30);
        M[k][k] += dt[k];
      }
      if (!spd6_inverse(M, Mi)) {
        for (int k = 0; k < 21; ++k) Mi[k] = 0.f;
        for (int k = 0; k < 6; ++k) Mi[sym6(k, k)] = M[k][k] > 0.0 ? (float)(1.0 / M[k][k]) : 0.f;
      }
      rp = mul(gp, -1.f);
      rw = mul(gw, -1.f);
      minv(rp, rw, zp, zw);
      zo = m9v(J, zw);
      dlp = dlw = pp = pw = qp = qw = make_float3(0.f, 0.f, 0.f);
      v[0] = dot3(rp, zp) + dot3(rw, zw);
      v[1] = dot3(rp, rp) + dot3(rw, rw);
    }
    scaled = true;
    publish(zp, zw, zo);
    team.template reduce<2, 0>(v);
    double rz = v[0];
    const double tol2 = (double)opt.pcg_relative_tolerance * opt.pcg_relative_tolerance * v[1];
    if (!(v[1] > 0.0)) return 0;
    float beta = 0.f;
    int k = 0;
    for (; k < opt.pcg_max_iterations; ++k) {
      stage();
      double v1[1] = {0.0};
      if (mine) {
        const float gd = dotf(g, zp);
        float3 ap = make_float3(0.f, 0.f, 0.f), aw = ap, tor = ap;
        for (int n = e0; n < e1; ++n) {
          const float4 le = LE[n];
          const unsigned pk = __float_as_uint(le.w);
          const float3 e = f3(le);
          float3 a, b, c;
          record(pk, a, b, c);
          const float mo = out_mult(pk), mi = in_mult(pk);
          const float3 d = sub(zp, a);
          const float3 y = add(d, cross3(zo, e));
          const float3 om = make_float3(mo * zo.x + mi * c.x, mo * zo.y + mi * c.y, mo * zo.z + mi * c.z);
          ap = add(ap, madd(cross3(om, e), mo + mi, d));
          aw = madd(aw, mo + mi, sub(zw, b));
          tor = madd(tor, mo, cross3(e, y));
        }
        tor = m9tv(J, tor);
        ap = make_float3(l2 * ap.x + g.x * gd + dt[0] * zp.x, l2 * ap.y + g.y * gd + dt[1] * zp.y,
                         l2 * ap.z + g.z * gd + dt[2] * zp.z);
        aw = make_float3(aw.x + l2 * tor.x + dt[3] * zw.x, aw.y + l2 * tor.y + dt[4] * zw.y,
                         aw.z + l2 * tor.z + dt[5] * zw.z);
        pp = madd(zp, beta, pp);
        pw = madd(zw, beta, pw);
        qp = madd(ap, beta, qp);
        qw = madd(aw, beta, qw);
        v1[0] = dot3(pp, qp) + dot3(pw, qw);
      }
      team.template reduce<1, 0>(v1);
      if (!(v1[0] > 0.0)) break;
      const float fa = (float)(rz / v1[0]);
      double v2[2] = {0.0, 0.0};
      if (mine) {
        dlp = madd(dlp, fa, pp);
        dlw = madd(dlw, fa, pw);
        rp = madd(rp, -fa, qp);
        rw = madd(rw, -fa, qw);
        minv(rp, rw, zp, zw);
        zo = m9v(J, zw);
        v2[0] = dot3(rp, zp) + dot3(rw, zw);
        v2[1] = dot3(rp, rp) + dot3(rw, rw);
      }
      publish(zp, zw, zo);
      team.template reduce<2, 0>(v2);
      beta = (float)(v2[0] / rz);
      rz = v2[0];
      if (v2[1] <= tol2) { ++k; break; }
    }
    return k;
  };

  // ---- model cost change, candidate cost, step and parameter norms ---------
  auto candidate = [&]() -> LMCandidate {
    publish(dlp, dlw, dlw);
    team.barrier();
    stage();
    double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (mine) {
      const float gd = dotf(g, dlp);
      v[0] = (double)gd * ((double)dist + 0.5 * (double)gd);
      const float dc = lookup_f32(P.grid, P.N, x0.x + (u.x + dlp.x), x0.y + (u.y + dlp.y), x0.z + (u.z + dlp.z));
      v[1] = 0.5 * (double)dc * (double)dc;
      v[3] = dot3(dlp, dlp) + dot3(dlw, dlw);
      const float3 x = add(x0, u);
      v[4] = dot3(x, x) + dot3(w, w);
      const float3 om = m9v(J, dlw);
      const float wv[3] = {w.x + dlw.x, w.y + dlw.y, w.z + dlw.z};
      float Am[9];
      rotation_point_jacobian(wv, Am);
      for (int n = e0; n < e1; ++n) {
        const float4 le = LE[n];
        const unsigned pk = __float_as_uint(le.w);
        const float mo = out_mult(pk);
        if (!(mo > 0.f)) continue;
        const float3 e = f3(le);
        float3 a, b, c;
        record(pk, a, b, c);
        const float3 d = sub(dlp, a), ms = sub(dlw, b);
        const float3 y = add(d, cross3(om, e));
        const float3 sg = f3(ES[n]);
        v[0] += (double)mo * (dot3(y, f3(ER[n])) + 0.5 * (double)l2 * dot3(y, y) + dot3(ms, madd(sg, 0.5f, ms)));
        const float3 rc = mul(sub(m9v(Am, add(e, d)), f3(EV[n])), lam);
        const float3 s2 = add(sg, ms);
        v[2] += 0.5 * (double)mo * (dot3(rc, rc) + dot3(s2, s2));
      }
    }
    team.template reduce<5, 0>(v);
    return LMCandidate{-v[0], v[1] + v[2], sqrt(v[3]), sqrt(v[4])};
  };
  auto accept = [&]() {
    u = add(u, dlp);
    w = add(w, dlw);
  };
  lm_trust_region_loop(opt, eval, solve, candidate, accept, team.leader() ? res + C.pid : nullptr, clock_start);
  if (mine) {
    A.u[vi] = f4(u);
    A.w[vi] = f4(w);
  }
}

}  // namespace

int lm_rot_launch(const RotPairDesc* pairs_dev, int npairs, const RotArrays& arrays, const LMOptionsDev& opt,
                  LMResultDev* results_dev, long long total_vertices, long long total_half_edges, int block_threads,
                  hipStream_t s) {
  if (npairs <= 0) return MO_OK;
  MO_CHECK(block_threads >= 64 && block_threads <= 256 && block_threads % 64 == 0, MO_ERR_ARG,
           "block_threads must be a multiple of 64 in [64, 256] (got %d)", block_threads);
  hipLaunchKernelGGL(k_lm_rot, dim3(npairs), dim3(block_threads), 0, s, pairs_dev, arrays, opt, results_dev,
                     total_vertices, total_half_edges);
  MO_HIP(hipGetLastError());
  return MO_OK;
}

// Bound on any one wait of a team, in device clock ticks.
static int team_wait_limit(long long* limit) {
  int dev = 0, khz = 0;
  MO_HIP(hipGetDevice(&dev));
  MO_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
  *limit = (long long)std::max(khz, 1) * 1000LL * 20;   // 20 s
  if (const char* w = getenv("MO_LM_TEAM_WAIT_US")) *limit = atoll(w) * (long long)std::max(khz, 1) / 1000LL;
  return MO_OK;
}

// MO_LM_COOP_REFUSE=k treats the call's k-th and later cooperative launches
// as refused without trying them (the fallback path's test hook; the
// runtime refuses cooperative grids while another process holds the GPU)
static bool refused_by_host(int coop) {
  const char* f = getenv("MO_LM_COOP_REFUSE");
  return f && atoi(f) > 0 && coop >= atoi(f);
}

int lm_rot_team_capacity(int block_threads) {
  int dev = 0, cus = 0, per = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void*)k_lm_rot_team, block_threads, 0) != hipSuccess)
    return 0;
  return per * cus;
}

int lm_rot_team_launch(const RotPairDesc* pairs_dev, const int* plist, const int4* wg_dev, int nwg,
                       const RotArrays& arrays, const LMOptionsDev& opt, LMResultDev* results_dev,
                       long long total_vertices, long long total_half_edges, int block_threads, int coop,
                       unsigned* cnt, double* part, int* abort_flag, hipStream_t s) {
  if (nwg <= 0) return MO_OK;
  MO_CHECK(block_threads >= 64 && block_threads <= 256 && block_threads % 64 == 0, MO_ERR_ARG,
           "block_threads must be a multiple of 64 in [64, 256] (got %d)", block_threads);
  long long limit = 0;
  if (int rc = team_wait_limit(&limit)) return rc;
  RotArrays a = arrays;
  LMOptionsDev o = opt;
  LMResultDev* r = results_dev;
  long long tv = total_vertices, th = total_half_edges;
  void* args[] = {(void*)&pairs_dev, (void*)&plist, (void*)&wg_dev, (void*)&a, (void*)&o, (void*)&r, (void*)&tv,
                  (void*)&th, (void*)&cnt, (void*)&part, (void*)&abort_flag, (void*)&limit};
  if (refused_by_host(coop)) return kCoopRefused;
  if (hipLaunchCooperativeKernel((const void*)k_lm_rot_team, dim3(nwg), dim3(block_threads), args, 0, s) !=
      hipSuccess) {
    (void)hipGetLastError();   // the runtime refused the cooperative grid: nothing was launched
    return kCoopRefused;
  }
  return MO_OK;
}

size_t lm_rot_chip_lds(int threads, int nhalo, int nent) {
  return 48 * ((size_t)threads + (size_t)nhalo) + 16 * (size_t)nent;
}

int lm_rot_chip_slot_words() { return kTagSlotWords; }

static const void* chip_kernel(int threads) {
  return threads == 256 ? (const void*)k_lm_rot_chip<256> : (const void*)k_lm_rot_chip<512>;
}

int lm_rot_chip_capacity(int threads, size_t lds_bytes) {
  int dev = 0, cus = 0, per = 0;
  if (hipFuncSetAttribute(chip_kernel(threads), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes) !=
          hipSuccess ||
      hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, chip_kernel(threads), threads, lds_bytes) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return per * cus;
}

int lm_rot_chip_launch(const RotPairDesc* pairs_dev, const RotChunk* chunks_dev, int nchunks, const RotChipArrays& a,
                       const LMOptionsDev& opt, LMResultDev* results_dev, int threads, size_t lds_bytes, int coop,
                       unsigned long long* slots, int* abort_flag, hipStream_t s) {
  if (nchunks <= 0) return MO_OK;
  MO_HIP(hipFuncSetAttribute(chip_kernel(threads), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes));
  long long limit = 0;
  if (int rc = team_wait_limit(&limit)) return rc;
  RotChipArrays arr = a;
  LMOptionsDev o = opt;
  void* args[] = {(void*)&pairs_dev, (void*)&chunks_dev, (void*)&arr,        (void*)&o,
                  (void*)&results_dev, (void*)&slots,    (void*)&abort_flag, (void*)&limit};
  if (!coop) {
    MO_HIP(hipLaunchKernel(chip_kernel(threads), dim3(nchunks), dim3(threads), args, lds_bytes, s));
    return MO_OK;
  }
  if (refused_by_host(coop)) return kCoopRefused;
  if (hipLaunchCooperativeKernel(chip_kernel(threads), dim3(nchunks), dim3(threads), args, (unsigned)lds_bytes, s) !=
      hipSuccess) {
    (void)hipGetLastError();   // the runtime refused the cooperative grid: nothing was launched
    return kCoopRefused;
  }
  return MO_OK;
}

}  // namespace mo
