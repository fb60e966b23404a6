// The adjoint of the fused right-hand side: the vector-Jacobian products of
// the pointwise algebra in the point's orthonormal frame (tgh_stage.hpp), of
// the closed-form Kerr-Schild gauge source and of the layer, written by hand,
// and the kernels that apply them on the brick layout:
//
//   k_adj_point   one evolved brick point per thread: the stage input's
//                 stencils and the cotangent of F at the point give the
//                 point's local cotangents -- of the point values (h, Pi), of
//                 the first derivatives of h and Pi, of the second derivatives
//                 of h and of the Kreiss-Oliger sums -- written to scratch
//                 fields, and the parameters' cotangent, folded per workgroup;
//   k_adj_gather  one evolved brick point per thread: the transposed stencils
//                 (the forward offsets reversed) gather the scratch fields into
//                 the cotangent of the stage input, and the RK4 combine's
//                 transpose forms the next stage's cotangent.
//
// The parameters differentiated are the constraint damping's Gaussian rates
// (gamma0_near, gamma0_far), gamma2, and the layer's rho_max and rho ramp
// fraction (the interior layer, src/interior.jl:178-238; the damping,
// src/gauge.jl:1094-1156). The reference has no adjoint: it differentiates
// nothing; the oracle's dual-number tangent of the same right-hand side is
// what pins these transposes (<lambda, J v> = <J^T lambda, v>).
#pragma once
#include "tgh_stage.hpp"

namespace tgh {

enum { ADJ_NPAR = 5 };  // gamma0_near, gamma0_far, gamma2, rho_max, rho_ramp

// ---------------------------------------------------------------------------
// The transpose of the pointwise algebra in the point's orthonormal frame
// (tgh_stage.hpp). The forward forms every quantity from tensors' frame
// components, T' = E T E^T with E = (n; e_A) the frame's matrix, and from E's
// own entries (alpha, beta, gamma^ij, sqrt(gamma)). A change of the metric
// changes E by Omega = dE E^-1, ten numbers (nn, nA and AB with A >= B: E is
// triangular), so the cotangents of all coefficients collapse into Omega's --
// a tensor's adds 2 T'bar T', alpha's -alpha to nn, and so on -- and Omega
// comes from the metric's change in the frame by
//   dg'_nn = 2 Omega_nn, dg'_nA = -Omega_nA, dg'_AB = -(Omega_AB + Omega_BA).
// Cotangents of symmetric tensors are held as the symmetric matrix F with
// <cotangent, T> = sum over all pairs of F_ab T_ab (packed, off-diagonal pairs
// counted twice), so that they transform as tensors do.
__device__ __forceinline__ constexpr double sym_mult(int n) { return prow(n) == pcol(n) ? 1.0 : 2.0; }

// F' = C^T F C: coordinate components' cotangent to the frame components',
// T = C T' C^T with d_t = alpha n + b_A e_A and d_i = L_iA e_A.
__device__ __forceinline__ void cot_to_frame(const Frame& f, double c[NC]) {
  double G[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const double t = c[pidx(a, 0)], x = c[pidx(a, 1)], y = c[pidx(a, 2)], z = c[pidx(a, 3)];
    G[a][0] = f.al * t;
    G[a][1] = f.b[0] * t + f.L11 * x + f.L21 * y + f.L31 * z;
    G[a][2] = f.b[1] * t + f.L22 * y + f.L32 * z;
    G[a][3] = f.b[2] * t + f.L33 * z;
  }
#pragma unroll
  for (int B = 0; B < 4; ++B) {
    if (B == 0) c[0] = f.al * G[0][0];
    if (B <= 1) c[pidx(1, B)] = f.b[0] * G[0][B] + f.L11 * G[1][B] + f.L21 * G[2][B] + f.L31 * G[3][B];
    if (B <= 2) c[pidx(2, B)] = f.b[1] * G[0][B] + f.L22 * G[2][B] + f.L32 * G[3][B];
    c[pidx(3, B)] = f.b[2] * G[0][B] + f.L33 * G[3][B];
  }
}
// F = E^T F' E, the other way.
__device__ __forceinline__ void cot_from_frame(const Frame& f, double c[NC]) {
  const double r0 = -f.ra * f.bu[0], r1 = -f.ra * f.bu[1], r2 = -f.ra * f.bu[2];
  double G[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const double n = c[pidx(a, 0)], p = c[pidx(a, 1)], q = c[pidx(a, 2)], s = c[pidx(a, 3)];
    G[a][0] = f.ra * n;
    G[a][1] = r0 * n + f.e11 * p + f.e21 * q + f.e31 * s;
    G[a][2] = r1 * n + f.e22 * q + f.e32 * s;
    G[a][3] = r2 * n + f.e33 * s;
  }
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    if (b == 0) c[0] = f.ra * G[0][0];
    if (b <= 1) c[pidx(1, b)] = r0 * G[0][b] + f.e11 * G[1][b] + f.e21 * G[2][b] + f.e31 * G[3][b];
    if (b <= 2) c[pidx(2, b)] = r1 * G[0][b] + f.e22 * G[2][b] + f.e32 * G[3][b];
    c[pidx(3, b)] = r2 * G[0][b] + f.e33 * G[3][b];
  }
}
// om += 2 s F T over Omega's entries (nn, nA, AB with A >= B, at pidx(A, B)).
__device__ __forceinline__ void add_omega(double om[NC], double s, const double F[NC], const double T[NC]) {
#pragma unroll
  for (int n = 0; n < NC; ++n) {
    // n = (a, c) with a >= c: Omega's entry (n, A) is row n, column A
    const int a = n < 4 ? 0 : prow(n), c = n < 4 ? n : pcol(n);
    double x = F[pidx(a, 0)] * T[pidx(0, c)];
#pragma unroll
    for (int b = 1; b < 4; ++b) x += F[pidx(a, b)] * T[pidx(b, c)];
    om[n] += 2.0 * s * x;
  }
}

// Twice the lowered Christoffels from the derivatives in place (frame_source's
// map, its own transpose in the symmetric convention above), and the inverse
// M_a[bc] = (G_b[ac] + G_c[ab]) / 2.
__device__ __forceinline__ void christoffel_map(double M[4][NC]) {
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = a + 1; b < 4; ++b) {
#pragma unroll
      for (int c = b + 1; c < 4; ++c) {
        double &x = M[a][pidx(b, c)], &y = M[b][pidx(a, c)], &z = M[c][pidx(a, b)];
        const double t = x + y + z;
        x = t - 2.0 * x;
        y = t - 2.0 * y;
        z = t - 2.0 * z;
      }
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        const int p = o ? b : a, q = o ? a : b;
        double &u = M[p][pidx(q, q)], &v = M[q][pidx(p, q)];
        const double t = u;
        u = 2.0 * v - u;
        v = t;
      }
    }
}
__device__ __forceinline__ void christoffel_unmap(double G[4][NC]) {
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = a + 1; b < 4; ++b) {
#pragma unroll
      for (int c = b + 1; c < 4; ++c) {
        double &x = G[a][pidx(b, c)], &y = G[b][pidx(a, c)], &z = G[c][pidx(a, b)];
        const double X = x, Y = y, Z = z;
        x = 0.5 * (Y + Z);
        y = 0.5 * (X + Z);
        z = 0.5 * (X + Y);
      }
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        const int p = o ? b : a, q = o ? a : b;
        double &u = G[p][pidx(q, q)], &v = G[q][pidx(p, q)];
        const double t = v;
        v = 0.5 * (u + v);
        u = t;
      }
    }
}

// frame_source and its transpose: from M (kept), H, wA, g0, g2 and Y, the
// cotangent of its result S: S itself, the cotangents of M (Mb), H and wA
// (set), and of g0 and g2 (added).
__device__ __forceinline__ void frame_source_vjp(double M[4][NC], const double H[4], const double wA[3], double g0,
                                                 double g2, const double Y[NC], double S[NC], double Mb[4][NC],
                                                 double Hb[4], double wb[3], double& g0b, double& g2b) {
  const double sg[4] = {-1.0, 1.0, 1.0, 1.0};
  double T[4], Tb[4] = {0.0, 0.0, 0.0, 0.0}, cf[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const double s = -M[0][pidx(c, 0)] + M[1][pidx(c, 1)] + M[2][pidx(c, 2)] + M[3][pidx(c, 3)];
    T[c] = s - 0.5 * ((M[c][4] + M[c][7] + M[c][9]) - M[c][0]);
    cf[c] = c == 0 ? 0.5 * T[0] : -0.5 * (T[c] + wA[c - 1]);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    // S += cf_e M_e + sum_c s_e s_c M_e[cA] M_e[cB], with N = M_e Y
    double cb = 0.0, N[4][4];
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      cb += sym_mult(n) * Y[n] * M[e][n];
      const int a = prow(n), b = pcol(n);
      double s = 0.0;
#pragma unroll
      for (int c = 0; c < 4; ++c) s += sg[e] * sg[c] * M[e][pidx(c, a)] * M[e][pidx(c, b)];
      S[n] = (e == 0 ? 0.0 : S[n]) + (s + cf[e] * M[e][n]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int A = 0; A < 4; ++A) {
        double s = 0.0;
#pragma unroll
        for (int B = 0; B < 4; ++B) s += M[e][pidx(c, B)] * Y[pidx(B, A)];
        N[c][A] = s;
      }
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      const int c = prow(n), A = pcol(n);
      Mb[e][n] = cf[e] * Y[n] + sg[e] * (sg[c] * N[c][A] + sg[A] * N[A][c]);
    }
    // cf_0 = T_0 / 2, cf_A = -(T_A + w_A) / 2
    Tb[e] += (e == 0 ? 0.5 : -0.5) * cb;
    if (e > 0) wb[e - 1] = -0.5 * cb;
  }
  christoffel_map(M);  // M holds G until unmapped
  double Gb[4][NC];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    // S += -GG / 4 + (s_a H_a / 2) G_a
    const double hh = 0.5 * sg[a] * H[a];
    double hb = 0.0;
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      hb += sym_mult(n) * Y[n] * M[a][n];
      S[n] += hh * M[a][n];
      double s = 0.0;
#pragma unroll
      for (int b = 0; b < 4; ++b) s += Y[pidx(a, b)] * M[b][n];
      Gb[a][n] = hh * Y[n] - 0.5 * sg[prow(n)] * sg[pcol(n)] * s;
    }
    Hb[a] = 0.5 * sg[a] * hb;
  }
#pragma unroll
  for (int n = 0; n < NC; ++n) {
    const int a = prow(n), b = pcol(n);
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < NC; ++q) s += sym_mult(q) * sg[prow(q)] * sg[pcol(q)] * M[a][q] * M[b][q];
    S[n] -= 0.25 * s;
  }
  christoffel_unmap(M);
  christoffel_map(Gb);
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int n = 0; n < NC; ++n) Mb[a][n] += Gb[a][n];
  // the damping
  {
    const double C0 = T[0] + H[0], C1 = T[1] + H[1], C2 = T[2] + H[2], C3 = T[3] + H[3];
    const double hg = 0.5 * g0, k1 = (1.0 + g2) * C0, Yd = Y[4] + Y[7] + Y[9];
    S[0] += hg * (k1 - 2.0 * C0);
    S[1] -= hg * C1;
    S[2] -= hg * C2;
    S[3] -= hg * C3;
    S[4] -= hg * k1;
    S[7] -= hg * k1;
    S[9] -= hg * k1;
    const double k1b = hg * (Y[0] - Yd);
    // off-diagonal S_nA: the packed entry counts twice
    const double Cb[4] = {(1.0 + g2) * k1b - 2.0 * hg * Y[0], -2.0 * hg * Y[1], -2.0 * hg * Y[2], -2.0 * hg * Y[3]};
    g2b += C0 * k1b;
    g0b += 0.5 * (Y[0] * (k1 - 2.0 * C0) - 2.0 * (Y[1] * C1 + Y[2] * C2 + Y[3] * C3) - k1 * Yd);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      Tb[c] += Cb[c];
      Hb[c] += Cb[c];
    }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      Mb[e][pidx(c, e)] += (c == e ? 1.0 : 0.5) * sg[e] * Tb[c];
      Mb[c][pidx(e, e)] -= 0.5 * sg[e] * Tb[c];
    }
}

// The reverse of ks_source (the closed-form Kerr-Schild gauge source of a
// hole at rest, spin along z): the cotangents of h (its tt, tx, ty, tz
// components) and of D[c] (the same components) from those of H_a and d_c H_a.
TGH_HD void ks_source_vjp(double M, double a, const double h[NC], const double D[4][NC], const double Hb[4],
                          const double Sb[NC], double hb[NC], double Db[4][NC]) {
  const double w[4] = {h[0], h[1], h[2], h[3]};
  const double K = w[0];
  const double sw = a * w[3];
  const double rad = M * M - sw * sw;
  const double root = rad > 0.0 ? sqrt(rad) : 0.0;
  const double Dn = M + root;
  const double iD = 1.0 / Dn;
  double wb[4] = {0.0, 0.0, 0.0, 0.0}, Kb = 0.0, iDb = 0.0, swb = 0.0, rootb = 0.0;
  // Hl[q] = -K iD w_q
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    wb[q] -= Hb[q] * K * iD;
    Kb -= Hb[q] * iD * w[q];
    iDb -= Hb[q] * K * w[q];
  }
  // dH[c][q] = -(dK w_q + K dw_q) iD + K w_q dD iD^2, dK = D[c][0], dD = -sw a D[c][3] / root
#pragma unroll
  for (int cc = 0; cc < 4; ++cc) {
    const double dK = D[cc][0];
    const double dD = root > 0.0 ? -sw * (a * D[cc][3]) / root : 0.0;
    double dKb = 0.0, dDb = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const double g = -(cc == q ? 2.0 : 1.0) * Sb[pidx(cc, q)];  // the cotangent of d_cc H_q
      const double dwq = D[cc][q];
      dKb -= g * w[q] * iD;
      wb[q] += -g * dK * iD + g * K * dD * iD * iD;
      Kb += -g * dwq * iD + g * w[q] * dD * iD * iD;
      Db[cc][q] -= g * K * iD;
      dDb += g * K * w[q] * iD * iD;
      iDb += -g * (dK * w[q] + K * dwq) + 2.0 * g * K * w[q] * dD * iD;
    }
    Db[cc][0] += dKb;
    if (root > 0.0) {
      Db[cc][3] += dDb * (-sw * a / root);
      swb += dDb * (-a * D[cc][3] / root);
      rootb += dDb * (sw * a * D[cc][3] / (root * root));
    }
  }
  rootb += -iDb * iD * iD;
  if (root > 0.0) swb += rootb * (-sw / root);
  wb[3] += a * swb;
  wb[0] += Kb;
#pragma unroll
  for (int q = 0; q < 4; ++q) hb[q] += wb[q];
}

// ---------------------------------------------------------------------------
// The scratch fields of one VJP (brick layout, zero on the frame): per
// variable v the cotangents of the point value h_v (AH) and Pi_v (AP), of the
// first derivatives d_i h_v (BH) and d_i Pi_v (BP) -- the scaled derivatives
// (1/h) st_d1 --, of the second derivatives of h_v in A's order xx, xy, xz,
// yy, yz, zz (CH, the mixed ones carrying the forward's factor 2), and of the
// Kreiss-Oliger sums of h_v (DH) and Pi_v (DP) with the amplitude over h
// folded in.
enum {
  AF_AH = 0,
  AF_AP = 10,
  AF_BH = 20,
  AF_BP = 50,
  AF_CH = 80,
  AF_DH = 140,
  AF_DP = 150,
  AF_N = 160
};

struct AdjPointArgs {
  Brick k;
  CaseP c;
  double t;
  const double* __restrict__ W;     // the stage input (brick, frame filled)
  const double* __restrict__ Hsrc;  // the sampled gauge source (brick) or null
  const double* __restrict__ kb;    // the cotangent of this stage's F (brick)
  double* __restrict__ F;           // AF_N scratch fields (brick)
  double* __restrict__ thp;         // ADJ_NPAR accumulators per logical workgroup
  const double* __restrict__ lbox;  // the layer's targets (RhsArgs::lbox)
  long lB3;
  int lB;
};

struct AdjGatherArgs {
  Brick k;
  const double* __restrict__ F;
  const double* __restrict__ lam;
  double* __restrict__ lacc;
  double* __restrict__ kbn;
  double* __restrict__ ybar;  // the VJP alone (tgh_vjp_rhs), or null
  double cl, cy;
  int first, last;
};
struct AdjInitArgs {
  Brick k;
  CaseP c;
  double t, J, nw, cl;
  const double* __restrict__ u;
  double* __restrict__ lam;
  double* __restrict__ kbn;
};
struct AdjCopiesArgs {
  Geom g;
  Brick k;
  const double* __restrict__ src;  // block layout
  double* __restrict__ dst;        // brick layout
};
// One evolved brick point: F(u) recomputed in the frame, then its transpose
// applied to the point's cotangent (lh for d_t h, lP for d_t Pi).
// What bounds it: a thousand loads and 160 stores a point, one wave a SIMD
// (the derivatives, their cotangents and the frame are 130 numbers). In
// coordinates, with the coefficients' cotangents held, it spilled 3 KB a lane:
// the VJP of 64 blocks of 16^3 took 2.10 ms, 0.94 with this and the gather below.
template <int Q, int GAUGE, int HOLE>
__device__ __forceinline__ void adj_point(const AdjPointArgs& a, int x, int y, int z, double th[ADJ_NPAR]) {
  const Brick& k = a.k;
  const CaseP& c = a.c;
  const long off = brick_index(k, x, y, z), fs = k.fs;
  const int sy = (int)k.py, sz = (int)k.pz;
  const double xp[3] = {grid_coord(k.lo[0], x, k.h), grid_coord(k.lo[1], y, k.h), grid_coord(k.lo[2], z, k.h)};
  double* __restrict__ F = a.F + off;
  double r = 0.0;
  if (frozen_core<HOLE>(c, a.t, xp, r)) {
    // a hole at rest: du = 0 in the core, whatever u holds
#pragma unroll 1
    for (int f = 0; f < AF_N; ++f) F[f * fs] = 0.0;
    return;
  }
  const double* __restrict__ w0 = a.W + off;
  const double* __restrict__ kb = a.kb + off;
  const double ih = k.inv_h, ih2 = ih * ih;
  const double epsh = c.has_diss ? dissipation_rate(c, a.t, xp) * ih : 0.0;
  // ---- forward: the derivatives, the frame ----
  double hv[NC], M[4][NC], Dk[4][NC];  // Dk: the coordinate derivatives of h_ta
#pragma unroll
  for (int v = 0; v < NC; ++v) {
    const double* __restrict__ pv = w0 + v * fs;
    hv[v] = pv[0];
    M[1][v] = ih * st_d1<Q>(pv, 1);
    M[2][v] = ih * st_d1<Q>(pv, sy);
    M[3][v] = ih * st_d1<Q>(pv, sz);
    M[0][v] = epsh * (st_ko<Q>(pv, 1) + st_ko<Q>(pv, sy) + st_ko<Q>(pv, sz));
#pragma unroll
    for (int d = 0; d < 4; ++d) asm volatile("" : "+v"(M[d][v]));
    __builtin_amdgcn_sched_barrier(0);
  }
  Frame f;
  make_frame(hv, f);
  const double as = f.al * f.sg;
#pragma unroll
  for (int v = 0; v < NC; ++v) {
    M[0][v] = w0[(NC + v) * fs] * f.isg + M[0][v] * f.ra;  // D_n h
    if (v < 4) {
      Dk[0][v] = f.bu[0] * M[1][v] + f.bu[1] * M[2][v] + f.bu[2] * M[3][v] + f.al * M[0][v];
#pragma unroll
      for (int d = 1; d < 4; ++d) Dk[d][v] = M[d][v];
    }
    const double d1 = M[1][v], d2 = M[2][v], d3 = M[3][v];
    M[1][v] = f.e11 * d1;
    M[2][v] = f.e21 * d1 + f.e22 * d2;
    M[3][v] = f.e31 * d1 + f.e32 * d2 + f.e33 * d3;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) to_frame(f, M[e]);
  double Hl[4] = {0.0, 0.0, 0.0, 0.0}, Hf[4] = {0.0, 0.0, 0.0, 0.0}, dHs[NC];
  constexpr bool HAS_H = gauge_has_source(GAUGE);
  if constexpr (HAS_H) {
    double dH[4][4];
    if constexpr (GAUGE == GAUGE_SAMPLED) {
      const double* __restrict__ Hp = a.Hsrc + off;
#pragma unroll
      for (int q = 0; q < 4; ++q) Hl[q] = Hp[q * fs];
#pragma unroll
      for (int n = 0; n < 16; ++n) dH[n % 4][n / 4] = Hp[(4 + n) * fs];
    } else {
      ks_source(c.bg.M, c.bg.a, hv, Dk, Hl, dH);
    }
#pragma unroll
    for (int n = 0; n < NC; ++n) dHs[n] = dH[prow(n)][pcol(n)] + dH[pcol(n)][prow(n)];
    Hf[0] = (Hl[0] - (f.bu[0] * Hl[1] + f.bu[1] * Hl[2] + f.bu[2] * Hl[3])) * f.ra;
    Hf[1] = f.e11 * Hl[1];
    Hf[2] = f.e21 * Hl[1] + f.e22 * Hl[2];
    Hf[3] = f.e31 * Hl[1] + f.e32 * Hl[2] + f.e33 * Hl[3];
  }
  double e_g = 0.0, g0 = c.g0;  // the Gaussian's exp(-r^2 / 2 w^2)
  if (c.damping != 0) {
    e_g = exp(-radius2(c, a.t, xp) / (2.0 * c.g0_width * c.g0_width));
    g0 = c.g0_far + (c.g0_near - c.g0_far) * e_g;
  }
  const double dn = M[1][1] + M[2][2] + M[3][3], divb = f.al * dn;
  double wA[3];
#pragma unroll
  for (int A = 0; A < 3; ++A)
    wA[A] = 0.5 * ((M[1 + A][4] + M[1 + A][7] + M[1 + A][9]) - M[1 + A][0]) -
            (M[1][pidx(1, 1 + A)] + M[2][pidx(2, 1 + A)] + M[3][pidx(3, 1 + A)]);
  // ---- the output's cotangent through the layer ----
  double wgt = 1.0, rho = 0.0, sl = 0.0, ss = 0.0, arg = 0.0, rhob = 0.0;
  const bool layer = HOLE && r < c.r1;
  const double* __restrict__ lb = nullptr;
  if (layer) {
    sl = (r - c.r0) / (c.r1 - c.r0);
    wgt = smoothstep(sl / c.w_ramp);
    arg = (1.0 - sl) / c.rho_ramp;
    ss = smoothstep(arg);
    rho = c.interior == INT_FROZEN ? 0.0 : c.rho_max * ss;
    lb = a.lbox + layer_slot(x, y, z, a.lB);
  }
  if (layer) {
#pragma unroll
    for (int v = 0; v < NC; ++v)
      rhob -= kb[(NC + v) * fs] * (w0[(NC + v) * fs] - lb[(NC + v) * a.lB3]) + kb[v * fs] * (hv[v] - lb[v * a.lB3]);
  }
  // ---- the principal part: beta^i d_i Pi + divb Pi + A^ij d_i d_j h + KO(Pi)
  // (d_i A^ij d_j h is in the source, as wA) ----
  double bb[3] = {0.0, 0.0, 0.0}, divbb = 0.0, Ab[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  {
    const double A[6] = {as * (f.e11 * f.e11 + f.e21 * f.e21 + f.e31 * f.e31),
                         2.0 * as * (f.e21 * f.e22 + f.e31 * f.e32),
                         2.0 * as * (f.e31 * f.e33),
                         as * (f.e22 * f.e22 + f.e32 * f.e32),
                         2.0 * as * (f.e32 * f.e33),
                         as * (f.e33 * f.e33)};
    // rolled: unrolled, the ten components' code would not fit the instruction cache
#pragma unroll 1
    for (int v = 0; v < NC; ++v) {
      const double* __restrict__ ph = w0 + v * fs;
      const double* __restrict__ pP = w0 + (NC + v) * fs;
      const double p_ = wgt * kb[(NC + v) * fs];  // the cotangent of the principal part and of the source
      bb[0] += p_ * (ih * st_d1<Q>(pP, 1));
      bb[1] += p_ * (ih * st_d1<Q>(pP, sy));
      bb[2] += p_ * (ih * st_d1<Q>(pP, sz));
      divbb += p_ * pP[0];
      Ab[0] += p_ * (ih2 * st_d2<Q>(ph, 1));
      Ab[1] += p_ * (ih2 * st_mixed<Q>(ph, 1, sy));
      Ab[2] += p_ * (ih2 * st_mixed<Q>(ph, 1, sz));
      Ab[3] += p_ * (ih2 * st_d2<Q>(ph, sy));
      Ab[4] += p_ * (ih2 * st_mixed<Q>(ph, sy, sz));
      Ab[5] += p_ * (ih2 * st_d2<Q>(ph, sz));
#pragma unroll
      for (int i = 0; i < 3; ++i) F[(AF_BP + 10 * i + v) * fs] = p_ * f.bu[i];
#pragma unroll
      for (int n = 0; n < 6; ++n) F[(AF_CH + 10 * n + v) * fs] = p_ * A[n];
      F[(AF_DP + v) * fs] = p_ * epsh;
    }
  }
  // ---- the source and its transpose ----
  double om[NC], Mb[4][NC], Hb[4], wb[3], g0b = 0.0, g2b = 0.0, asb = 0.0, pb[NC];
#pragma unroll
  for (int n = 0; n < NC; ++n) pb[n] = wgt * kb[(NC + n) * fs];
#pragma unroll
  for (int n = 0; n < NC; ++n) om[n] = 0.0;
  {
    double Y[NC], S[NC];
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      Y[n] = (sym_mult(n) == 1.0 ? 1.0 : 0.5) * pb[n];
      if (HAS_H) asb += pb[n] * dHs[n];
    }
    cot_to_frame(f, Y);
    // out = alpha sqrt(gamma) (-2 S + dHs) in coordinates
#pragma unroll
    for (int n = 0; n < NC; ++n) Y[n] *= -2.0 * as;
    frame_source_vjp(M, Hf, wA, g0, c.g2, Y, S, Mb, Hb, wb, g0b, g2b);
    add_omega(om, -1.0, Y, S);
    double ys = 0.0;
#pragma unroll
    for (int n = 0; n < NC; ++n) ys += sym_mult(n) * Y[n] * S[n];
    asb += ys / as;
  }
  // wA and divb = alpha sum_A D_A g_nA
#pragma unroll
  for (int A = 0; A < 3; ++A) {
    Mb[1 + A][0] -= 0.5 * wb[A];
    Mb[1 + A][4] += 0.5 * wb[A];
    Mb[1 + A][7] += 0.5 * wb[A];
    Mb[1 + A][9] += 0.5 * wb[A];
#pragma unroll
    for (int B = 0; B < 3; ++B) Mb[1 + B][pidx(1 + B, 1 + A)] -= (A == B ? 1.0 : 0.5) * wb[A];
    Mb[1 + A][pidx(0, 1 + A)] += 0.5 * f.al * divbb;
  }
  om[0] -= f.al * dn * divbb;
  // A^ij = alpha sqrt(gamma) e_Ai e_Aj: X = e Ab e^T
  {
    const double a00 = Ab[0], a01 = Ab[1], a02 = Ab[2], a11 = Ab[3], a12 = Ab[4], a22 = Ab[5];
    const double t11 = f.e11 * a00, t12 = f.e11 * a01, t13 = f.e11 * a02;
    const double t21 = f.e21 * a00 + f.e22 * a01, t22 = f.e21 * a01 + f.e22 * a11, t23 = f.e21 * a02 + f.e22 * a12;
    const double t31 = f.e31 * a00 + f.e32 * a01 + f.e33 * a02, t32 = f.e31 * a01 + f.e32 * a11 + f.e33 * a12,
                 t33 = f.e31 * a02 + f.e32 * a12 + f.e33 * a22;
    const double x11 = t11 * f.e11, x21 = t21 * f.e11, x31 = t31 * f.e11;
    const double x22 = t21 * f.e21 + t22 * f.e22, x32 = t31 * f.e21 + t32 * f.e22;
    const double x33 = t31 * f.e31 + t32 * f.e32 + t33 * f.e33;
    (void)t12;
    (void)t13;
    (void)t23;
    om[4] += 2.0 * as * x11;
    om[5] += 2.0 * as * x21;
    om[6] += 2.0 * as * x31;
    om[7] += 2.0 * as * x22;
    om[8] += 2.0 * as * x32;
    om[9] += 2.0 * as * x33;
    asb += x11 + x22 + x33;
  }
  // alpha sqrt(gamma): d = -alpha sqrt(gamma) (Omega_nn + tr Omega_AB)
  om[0] -= as * asb;
  om[4] -= as * asb;
  om[7] -= as * asb;
  om[9] -= as * asb;
  // beta^i (of the principal part): d beta^i = -alpha Omega_nA e_Ai
  om[1] -= f.al * (f.e11 * bb[0]);
  om[2] -= f.al * (f.e21 * bb[0] + f.e22 * bb[1]);
  om[3] -= f.al * (f.e31 * bb[0] + f.e32 * bb[1] + f.e33 * bb[2]);
  // the gauge source
  double Db[4][NC], aH[NC];  // the cotangents of d_a h_tb and h_ta from it
#pragma unroll
  for (int v = 0; v < 4; ++v) {
#pragma unroll
    for (int d = 0; d < 4; ++d) Db[d][v] = 0.0;
    aH[v] = 0.0;
  }
  if constexpr (HAS_H) {
#pragma unroll
    for (int n = 0; n < NC; ++n) {  // Hf = E Hl: Omega's entry (a, c) takes Hb_a Hf_c
      const int p = n < 4 ? 0 : prow(n), q = n < 4 ? n : pcol(n);
      om[n] += Hb[p] * Hf[q];
    }
    if constexpr (GAUGE == GAUGE_KS) {
      const double rn = f.ra * Hb[0];
      const double Hlb[4] = {rn, f.e11 * Hb[1] + f.e21 * Hb[2] + f.e31 * Hb[3] - rn * f.bu[0],
                             f.e22 * Hb[2] + f.e32 * Hb[3] - rn * f.bu[1], f.e33 * Hb[3] - rn * f.bu[2]};
      double Sb[NC];  // ks_source_vjp's convention: dH_ab + dH_ba enters with a minus sign
#pragma unroll
      for (int n = 0; n < NC; ++n) Sb[n] = -as * pb[n];
      ks_source_vjp(c.bg.M, c.bg.a, hv, Dk, Hlb, Sb, aH, Db);
    }
  }
  // ---- d_t h = beta^i d_i h + alpha D_n h; D_n h = Pi / sqrt(gamma) + KO / alpha ----
#pragma unroll
  for (int e = 0; e < 4; ++e) add_omega(om, 1.0, Mb[e], M[e]);
#pragma unroll
  for (int A = 1; A < 4; ++A)  // the derivative's own index: D_A turns with Omega_AB
#pragma unroll
    for (int B = 1; B <= A; ++B) {
      double s = 0.0;
#pragma unroll
      for (int n = 0; n < NC; ++n) s += sym_mult(n) * Mb[A][n] * M[B][n];
      om[pidx(A, B)] += s;
    }
  {
    double d0b[NC], Y[NC];
#pragma unroll
    for (int v = 0; v < NC; ++v) {
      d0b[v] = wgt * kb[v * fs];
      if (v < 4) d0b[v] += Db[0][v];
      Y[v] = (sym_mult(v) == 1.0 ? 1.0 : 0.5) * d0b[v];
    }
    cot_to_frame(f, Y);
#pragma unroll
    for (int A = 1; A < 4; ++A) {
      double s = 0.0;
#pragma unroll
      for (int n = 0; n < NC; ++n) s += sym_mult(n) * Y[n] * M[A][n];
      om[A] -= f.al * s;
    }
    from_frame(f, M[0]);  // D_n h in coordinates again
    cot_from_frame(f, Mb[0]);
    double onn = 0.0, oss = 0.0;
#pragma unroll
    for (int v = 0; v < NC; ++v) {
      const double nb = sym_mult(v) * Mb[0][v] + f.al * d0b[v];
      const double pi_ = w0[(NC + v) * fs] * f.isg;
      onn += nb * (M[0][v] - pi_) - f.al * d0b[v] * M[0][v];
      oss += nb * pi_;
      const double lP = kb[(NC + v) * fs];
      F[(AF_AP + v) * fs] = nb * f.isg + (wgt * divb - rho) * lP;
      F[(AF_DH + v) * fs] = nb * f.ra * epsh;
    }
    om[0] += onn;
    om[4] += oss;
    om[7] += oss;
    om[9] += oss;
#pragma unroll
    for (int A = 1; A < 4; ++A) cot_from_frame(f, Mb[A]);
#pragma unroll
    for (int v = 0; v < NC; ++v) {
      const double m = sym_mult(v);
      const double n1 = m * Mb[1][v] + f.b[0] * d0b[v], n2 = m * Mb[2][v] + f.b[1] * d0b[v],
                   n3 = m * Mb[3][v] + f.b[2] * d0b[v];
      const double k1 = v < 4 ? Db[1][v] : 0.0, k2 = v < 4 ? Db[2][v] : 0.0, k3 = v < 4 ? Db[3][v] : 0.0;
      F[(AF_BH + v) * fs] = k1 + f.e11 * n1 + f.e21 * n2 + f.e31 * n3;
      F[(AF_BH + 10 + v) * fs] = k2 + f.e22 * n2 + f.e32 * n3;
      F[(AF_BH + 20 + v) * fs] = k3 + f.e33 * n3;
    }
  }
  // ---- Omega back to the metric ----
#pragma unroll
  for (int n = 0; n < NC; ++n) om[n] *= n == 0 ? 0.5 : -0.5;
  cot_from_frame(f, om);
#pragma unroll
  for (int v = 0; v < NC; ++v) {
    double e = sym_mult(v) * om[v] - rho * kb[v * fs];
    if (v < 4) e += aH[v];
    F[(AF_AH + v) * fs] = e;
  }
  // the parameters: gamma0 = far + (near - far) e; rho = rho_max s(arg)
  if (c.damping != 0) {
    th[0] += g0b * e_g;
    th[1] += g0b * (1.0 - e_g);
  }
  th[2] += g2b;
  if (layer && c.interior != INT_FROZEN) {
    th[3] += rhob * ss;
    const double u0 = fmin(fmax(arg, 0.0), 1.0);
    const double dss = (arg > 0.0 && arg < 1.0) ? 30.0 * u0 * u0 * (1.0 - u0) * (1.0 - u0) : 0.0;
    th[4] += rhob * c.rho_max * dss * (-(1.0 - sl) / (c.rho_ramp * c.rho_ramp));
  }
}

#ifdef TGH_ADJOINT_KERNELS  // the kernels: built in the adjoint's translation unit
template <int Q, int GAUGE, int HOLE>
__global__ __launch_bounds__(256) void k_adj_point(AdjPointArgs a) {
  const int total = brick_runs(a.k);
  const int L = wg_logical(total);
  if (L >= total) return;
  double th[ADJ_NPAR] = {0.0, 0.0, 0.0, 0.0, 0.0};
  int x, y, z;
  if (brick_run(a.k, L, x, y, z)) adj_point<Q, GAUGE, HOLE>(a, x, y, z, th);
  __shared__ double sh[ADJ_NPAR][256];
  const int tid = threadIdx.x;
#pragma unroll
  for (int q = 0; q < ADJ_NPAR; ++q) sh[q][tid] = th[q];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (tid < w)
#pragma unroll
      for (int q = 0; q < ADJ_NPAR; ++q) sh[q][tid] += sh[q][tid + w];
    __syncthreads();
  }
  if (tid < ADJ_NPAR) a.thp[(long)L * ADJ_NPAR + tid] += sh[tid][0];
}

// The transposed stencils at one evolved brick point q and one variable pair
// (blockIdx.y), and the RK4 combine's transpose: ybar = the cotangent of the
// stage input at q; then
//   lacc = (first ? lam : lacc) + ybar,  kbn = cl * lam + cy * ybar
// or, with last (the step's first stage, reversed last), kbn = cl * lacc.
// A shift by -o along an axis is an index difference, wrapped on a periodic
// axis (its frame holds copies of the points the shift lands on); on a
// Dirichlet axis the frame's scratch fields are zero.
// What bounds it: 133 loads a pair from the L2 (the fields of 64 blocks of
// 16^3, 350 MB, do not fit one XCD's); a thread per point ran the ten pairs one
// after another, four waves a SIMD in all, and formed each index by division:
// 0.48 ms a stage there.
template <int Q>
__global__ __launch_bounds__(256) void k_adj_gather(AdjGatherArgs a) {
  const Brick& k = a.k;
  int x, y, z;
  if (!brick_map(k, x, y, z)) return;
  const int v = blockIdx.y;
  constexpr int R = W<Q>::R, H = R + 1;
  const long off = brick_index(k, x, y, z), fs = k.fs;
  const double ih = k.inv_h, ih2 = ih * ih;
  const double* __restrict__ F = a.F + off;
  int sh[3][2 * H + 1];  // the index difference of a shift by -(m - H)
  {
    const int p[3] = {x, y, z}, st[3] = {1, (int)k.py, (int)k.pz};
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int m = 0; m < 2 * H + 1; ++m) {
        int o = H - m;
        if (k.periodic[d]) {
          if (p[d] + o < 0) o += k.n[d];
          else if (p[d] + o >= k.n[d]) o -= k.n[d];
        }
        sh[d][m] = o * st[d];
      }
  }
  double s1h = 0.0, s1P = 0.0, s2 = 0.0, sk = 0.0, skP = 0.0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double* __restrict__ bh = F + (AF_BH + 10 * d + v) * fs;
    const double* __restrict__ bp = F + (AF_BP + 10 * d + v) * fs;
    const double* __restrict__ ch = F + (AF_CH + 10 * sidx3(d, d) + v) * fs;
    const double* __restrict__ dh = F + (AF_DH + v) * fs;
    const double* __restrict__ dp = F + (AF_DP + v) * fs;
#pragma unroll
    for (int m = 0; m < 2 * R + 1; ++m) {
      const int i = sh[d][m + 1];
      if (m != R) {
        s1h += W<Q>::d1[m] * bh[i];
        s1P += W<Q>::d1[m] * bp[i];
      }
      s2 += W<Q>::d2[m] * ch[i];
    }
#pragma unroll
    for (int m = 0; m < 2 * R + 3; ++m) {
      sk += W<Q>::ko[m] * dh[sh[d][m]];
      skP += W<Q>::ko[m] * dp[sh[d][m]];
    }
  }
  // the mixed derivatives, outer axis d1 < inner axis d2 as the forward
#pragma unroll
  for (int pq = 0; pq < 3; ++pq) {
    const int d1 = pq == 2 ? 1 : 0, d2 = pq == 0 ? 1 : 2;
    const double* __restrict__ ch = F + (AF_CH + 10 * sidx3(d1, d2) + v) * fs;
#pragma unroll
    for (int m1 = 0; m1 < 2 * R + 1; ++m1) {
      if (m1 == R) continue;
      double inner = 0.0;
#pragma unroll
      for (int m2 = 0; m2 < 2 * R + 1; ++m2)
        if (m2 != R) inner += W<Q>::d1[m2] * ch[sh[d1][m1 + 1] + sh[d2][m2 + 1]];
      s2 += W<Q>::d1[m1] * inner;
    }
  }
  const double yb[2] = {F[(AF_AH + v) * fs] + (ih * s1h + ih2 * s2 + sk), F[(AF_AP + v) * fs] + (ih * s1P + skP)};
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const long idx = off + (v + NC * q) * fs;
    if (a.ybar) {
      a.ybar[idx] = yb[q];
      continue;
    }
    const double la = (a.first ? a.lam[idx] : a.lacc[idx]) + yb[q];
    a.lacc[idx] = la;
    a.kbn[idx] = a.last ? a.cl * la : a.cl * a.lam[idx] + a.cy * yb[q];
  }
}

// lambda_T = dJ/du_T for J = the masked L2 error sqrt(sum e^2 / nw) over the
// evolved brick points (r >= r_1; each brick point one primary, weight 1),
// and kbn = c lambda_T (the last stage's cotangent).
template <bool MOVE>
__global__ __launch_bounds__(256) void k_adj_init(AdjInitArgs a) {
  const Brick& k = a.k;
  int x, y, z;
  if (!brick_map(k, x, y, z)) return;
  const long off = brick_index(k, x, y, z), fs = k.fs;
  const double xp[3] = {k.lo[0] + (double)x * k.h, k.lo[1] + (double)y * k.h, k.lo[2] + (double)z * k.h};
  const bool keep = is_evolved(a.c, a.t, xp);
  double s[20];
  if (keep) case_state_any<MOVE ? BGS_ALL : BGS_STATIC>(a.c, a.t, xp, s);
  const double f = (a.J > 0.0 && a.nw > 0.0) ? 1.0 / (a.J * a.nw) : 0.0;
  for (int v = 0; v < 20; ++v) {
    const double l = keep ? (a.u[off + v * fs] - s[v]) * f : 0.0;
    a.lam[off + v * fs] = l;
    a.kbn[off + v * fs] = a.cl * l;
  }
}

// A block-layout cotangent summed over the copies of each brick point (a
// point on a block face is an own point of every block holding it, and each
// copy's F is the brick point's), into the brick.
__global__ __launch_bounds__(256) void k_adj_fold_copies(AdjCopiesArgs a) {
  const Brick& k = a.k;
  const Geom& g = a.g;
  int x, y, z;
  if (!brick_map(k, x, y, z)) return;
  const int gp[3] = {x, y, z};
  int nc[3], ob[3][2], lc[3][2];
  for (int d = 0; d < 3; ++d) {
    nc[d] = 0;
    const int o = gp[d] / g.N, l = gp[d] - o * g.N;
    if (o < g.nb[d]) {
      ob[d][nc[d]] = o;
      lc[d][nc[d]++] = l;
    }
    if (l == 0) {
      if (o > 0) {
        ob[d][nc[d]] = o - 1;
        lc[d][nc[d]++] = g.N;
      } else if (g.periodic[d]) {
        ob[d][nc[d]] = g.nb[d] - 1;
        lc[d][nc[d]++] = g.N;
      }
    }
  }
  const long psz = (long)g.P * g.P * g.P, off = brick_index(k, x, y, z);
  double val[20];
#pragma unroll
  for (int v = 0; v < 20; ++v) val[v] = 0.0;
  for (int i = 0; i < nc[0]; ++i)
    for (int j = 0; j < nc[1]; ++j)
      for (int m = 0; m < nc[2]; ++m) {
        const int b = g.lookup[ob[0][i] + g.nb[0] * (ob[1][j] + g.nb[1] * ob[2][m])];
        const double* src = a.src + (long)b * 20 * psz + lc[0][i] + (long)g.P * (lc[1][j] + (long)g.P * lc[2][m]);
#pragma unroll
        for (int v = 0; v < 20; ++v) val[v] += src[v * psz];
      }
#pragma unroll
  for (int v = 0; v < 20; ++v) a.dst[off + v * k.fs] = val[v];
}
// A brick cotangent onto the block layout's primaries (the copies, which the
// fill overwrites before every evaluation, take zero); dst is zeroed first.
__global__ __launch_bounds__(256) void k_adj_to_primaries(AdjCopiesArgs a) {
  const Brick& k = a.k;
  const Geom& g = a.g;
  int x, y, z;
  if (!brick_map(k, x, y, z)) return;
  const int gp[3] = {x, y, z};
  int loc[3];
  const int b = brick_primary(g, gp, loc);
  const long psz = (long)g.P * g.P * g.P, off = brick_index(k, x, y, z);
  double* d = a.dst + (long)b * 20 * psz + loc[0] + (long)g.P * (loc[1] + (long)g.P * loc[2]);
  double val[20];
#pragma unroll
  for (int v = 0; v < 20; ++v) val[v] = a.src[off + v * k.fs];
#pragma unroll
  for (int v = 0; v < 20; ++v) d[v * psz] = val[v];
}

#endif  // TGH_ADJOINT_KERNELS

}  // namespace tgh
