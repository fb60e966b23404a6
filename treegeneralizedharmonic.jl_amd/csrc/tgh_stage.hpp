// One RK4 stage's right-hand side in one kernel (the stepper's default form):
// a workgroup takes a tile of points, evaluates the head at one point per
// thread in an orthonormal frame, keeps the Pi components' coefficients in
// registers and LDS, and then forms the ten Pi components from LDS.
//
// Why one kernel: as two (k_brick_head, k_brick_pi) the 25 coefficients of a
// point cross memory twice (400 of the 1360 bytes a point moved per stage),
// and the head, whose coordinate-basis algebra held 392 registers, ran one
// wave per SIMD and waited on its own latency 65 % of the time. In the frame
// the head needs 256 registers, so two waves share a SIMD, and two thirds of
// the instructions. On the Kerr-Schild hole's 257^3 points (q = 4) a stage
// takes 5.1 to 6.7 ms (its epilogue reads 0 to 3 values a variable), where
// the two kernels took 8.2 + 5.0; the step 24 ms against 53.
// What bounds it: the vector unit and the LDS pipe are each busy 1.7 ms of a
// stage and the L1 1.1, which two waves a SIMD overlap only in part.
#pragma once
#include "tgh_kernels.hpp"

namespace tgh {

// 1/sqrt(x) to the last bits: the hardware's estimate (relative error below
// 2^-23) and one third-order correction, y (1 + e/2 + 3 e^2/8) with e = 1 - x y^2.
__device__ __forceinline__ double rsqrt_refined(double x) {
#pragma clang fp contract(off)
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

// Sums of products in one order: every multiply-add of the stage is written
// out and contraction is off, so that its kernels (one problem's, a batch's, a
// block's) round alike whatever the compiler would have contracted.
__device__ __forceinline__ double dot2(double a, double b, double c, double d) {
#pragma clang fp contract(off)
  return fma(a, b, c * d);
}
__device__ __forceinline__ double dot3(double a, double b, double c, double d, double e, double f) {
#pragma clang fp contract(off)
  return fma(a, b, fma(c, d, e * f));
}
// smoothstep, dissipation_rate and damping_rate so written.
__device__ __forceinline__ double smoothstep_stage(double s) {
#pragma clang fp contract(off)
  const double u = fmin(fmax(s, 0.0), 1.0);
  const double v = u * u * u * fma(u, fma(6.0, u, -15.0), 10.0);
  return fmin(fmax(v, 0.0), 1.0);
}
__device__ __forceinline__ double radius2(const CaseP& c, double t, const double x[3]) {
#pragma clang fp contract(off)
  double cc[3];
  center_at(c, t, cc);
  const double d1 = x[0] - cc[0], d2 = x[1] - cc[1], d3 = x[2] - cc[2];
  return dot3(d1, d1, d2, d2, d3, d3);
}
__device__ __forceinline__ double damping_stage(const CaseP& c, double r2) {
#pragma clang fp contract(off)
  if (c.damping == 0) return c.g0;
  return fma(c.g0_near - c.g0_far, exp(-r2 / (2.0 * c.g0_width * c.g0_width)), c.g0_far);
}
__device__ __forceinline__ double dissipation_stage(const CaseP& c, double r2) {
#pragma clang fp contract(off)
  if (c.diss == 0) return c.eps_ko;
  const double r = sqrt(r2);
  if (r >= c.eps_rh) return c.eps_ko;
  if (r <= c.eps_r1) return c.eps_in;
  return fma(c.eps_in - c.eps_ko, smoothstep_stage((c.eps_rh - r) / (c.eps_rh - c.eps_r1)), c.eps_ko);
}

// The orthonormal frame of a point: the unit normal n = (d_t - beta^i d_i)/alpha
// and the triad e_A = sum_i e_Ai d_i from the Cholesky factor of the spatial
// metric, gamma = L L^T, e = L^-1 (both lower triangular), so that
// gamma^ij = sum_A e_Ai e_Aj. In the frame the metric is diag(-1, 1, 1, 1) and
// raising an index costs a sign.
struct Frame {
  double e11, e21, e22, e31, e32, e33;
  double L11, L21, L22, L31, L32, L33;
  double b[3];          // beta in the triad, b_A = e_Ai beta_i
  double bu[3];         // beta^i
  double al, ra;        // alpha, 1/alpha
  double sg, isg;       // sqrt(det gamma) and its inverse
};
__device__ __forceinline__ void make_frame(const double h[NC], Frame& f) {
#pragma clang fp contract(off)
  const double gxx = 1.0 + h[4], gyy = 1.0 + h[7], gzz = 1.0 + h[9];
  f.e11 = rsqrt_refined(gxx);
  f.L11 = gxx * f.e11;
  f.L21 = h[5] * f.e11;
  f.L31 = h[6] * f.e11;
  const double d2 = fma(-f.L21, f.L21, gyy);
  f.e22 = rsqrt_refined(d2);
  f.L22 = d2 * f.e22;
  f.L32 = fma(-f.L31, f.L21, h[8]) * f.e22;
  const double d3 = fma(-f.L32, f.L32, fma(-f.L31, f.L31, gzz));
  f.e33 = rsqrt_refined(d3);
  f.L33 = d3 * f.e33;
  f.e21 = -(f.L21 * f.e11) * f.e22;
  f.e32 = -(f.L32 * f.e22) * f.e33;
  f.e31 = -dot2(f.L31, f.e11, f.L32, f.e21) * f.e33;
  f.sg = f.L11 * f.L22 * f.L33;
  f.isg = f.e11 * f.e22 * f.e33;
  f.b[0] = f.e11 * h[1];
  f.b[1] = dot2(f.e21, h[1], f.e22, h[2]);
  f.b[2] = dot3(f.e31, h[1], f.e32, h[2], f.e33, h[3]);
  f.bu[0] = dot3(f.e11, f.b[0], f.e21, f.b[1], f.e31, f.b[2]);
  f.bu[1] = dot2(f.e22, f.b[1], f.e32, f.b[2]);
  f.bu[2] = f.e33 * f.b[2];
  const double a2 = (1.0 - h[0]) + dot3(f.b[0], f.b[0], f.b[1], f.b[1], f.b[2], f.b[2]);
  f.ra = rsqrt_refined(a2);
  f.al = a2 * f.ra;
}

// A symmetric covariant tensor's packed components into the frame, in place:
// (tt, ti, ij) -> (nn, nA, AB).
__device__ __forceinline__ void to_frame(const Frame& f, double m[NC]) {
#pragma clang fp contract(off)
  const double q1 = m[1] - dot3(f.bu[0], m[4], f.bu[1], m[5], f.bu[2], m[6]);
  const double q2 = m[2] - dot3(f.bu[0], m[5], f.bu[1], m[7], f.bu[2], m[8]);
  const double q3 = m[3] - dot3(f.bu[0], m[6], f.bu[1], m[8], f.bu[2], m[9]);
  m[0] = (m[0] - dot3(f.bu[0], m[1] + q1, f.bu[1], m[2] + q2, f.bu[2], m[3] + q3)) * (f.ra * f.ra);
  const double n1 = q1 * f.ra, n2 = q2 * f.ra, n3 = q3 * f.ra;
  m[1] = f.e11 * n1;
  m[2] = dot2(f.e21, n1, f.e22, n2);
  m[3] = dot3(f.e31, n1, f.e32, n2, f.e33, n3);
  const double t11 = f.e11 * m[4];
  const double t21 = dot2(f.e21, m[4], f.e22, m[5]);
  const double t22 = dot2(f.e21, m[5], f.e22, m[7]);
  const double t31 = dot3(f.e31, m[4], f.e32, m[5], f.e33, m[6]);
  const double t32 = dot3(f.e31, m[5], f.e32, m[7], f.e33, m[8]);
  const double t33 = dot3(f.e31, m[6], f.e32, m[8], f.e33, m[9]);
  m[4] = f.e11 * t11;
  m[5] = f.e11 * t21;
  m[6] = f.e11 * t31;
  m[7] = dot2(f.e21, t21, f.e22, t22);
  m[8] = dot2(f.e21, t31, f.e22, t32);
  m[9] = dot3(f.e31, t31, f.e32, t32, f.e33, t33);
}
// And back: d_i = sum_A L_iA e_A, d_t = alpha n + sum_A b_A e_A.
__device__ __forceinline__ void from_frame(const Frame& f, double s[NC]) {
#pragma clang fp contract(off)
  const double t1 = fma(f.al, s[1], dot3(f.b[0], s[4], f.b[1], s[5], f.b[2], s[6]));
  const double t2 = fma(f.al, s[2], dot3(f.b[0], s[5], f.b[1], s[7], f.b[2], s[8]));
  const double t3 = fma(f.al, s[3], dot3(f.b[0], s[6], f.b[1], s[8], f.b[2], s[9]));
  s[0] = fma(f.al, fma(f.al, s[0], dot3(f.b[0], s[1], f.b[1], s[2], f.b[2], s[3])),
             dot3(f.b[0], t1, f.b[1], t2, f.b[2], t3));
  s[1] = f.L11 * t1;
  s[2] = dot2(f.L21, t1, f.L22, t2);
  s[3] = dot3(f.L31, t1, f.L32, t2, f.L33, t3);
  const double u11 = f.L11 * s[4];
  const double u21 = dot2(f.L21, s[4], f.L22, s[5]);
  const double u22 = dot2(f.L21, s[5], f.L22, s[7]);
  const double u31 = dot3(f.L31, s[4], f.L32, s[5], f.L33, s[6]);
  const double u32 = dot3(f.L31, s[5], f.L32, s[7], f.L33, s[8]);
  const double u33 = dot3(f.L31, s[6], f.L32, s[8], f.L33, s[9]);
  s[4] = f.L11 * u11;
  s[5] = f.L11 * u21;
  s[6] = f.L11 * u31;
  s[7] = dot2(f.L21, u21, f.L22, u22);
  s[8] = dot2(f.L21, u31, f.L22, u32);
  s[9] = dot3(f.L31, u31, f.L32, u32, f.L33, u33);
}

// Half of the source S0 + Z of gh_source without the gauge source's
// derivative, in the frame: M[E] = D_E g packed in the frame (E = n, 1, 2, 3),
// H the gauge source in the frame, g0 and g2 the damping's rates; and half of
// -wA^C D_C g, the flux's d_i (alpha sqrt(gamma) gamma^ij) d_j h over -alpha
// sqrt(gamma). M is overwritten (the lowered Christoffels take its place).
//   C2 + C2^T - 2 Gamma^c_da Gamma^d_cb = 2 g^cd g^ef (d_e g_ca d_f g_db - Gamma_ace Gamma_bdf)
// (both sides are products of d g with the antisymmetric and symmetric parts
// of its first two indices), which in the frame are sums of squares' products
// with signs: 160 + 100 multiplications where the coordinate form's raised
// tensors take 1100.
__device__ __forceinline__ void frame_source(double M[4][NC], const double H[4], const double wA[3], double g0,
                                             double g2, double S[NC]) {
#pragma clang fp contract(off)
  // Gamma_C = eta^EF Gamma_C,EF
  double T[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const double s = -M[0][pidx(c, 0)] + M[1][pidx(c, 1)] + M[2][pidx(c, 2)] + M[3][pidx(c, 3)];
    T[c] = fma(-0.5, (M[c][4] + M[c][7] + M[c][9]) - M[c][0], s);
  }
  const double C0 = T[0] + H[0], C1 = T[1] + H[1], C2 = T[2] + H[2], C3 = T[3] + H[3];
  const double hT0 = 0.5 * T[0], hT1 = 0.5 * (T[1] + wA[0]), hT2 = 0.5 * (T[2] + wA[1]), hT3 = 0.5 * (T[3] + wA[2]);
#pragma unroll
  for (int n = 0; n < NC; ++n) {
    const int a = prow(n), b = pcol(n);
    double s = fma(-hT3, M[3][n], fma(-hT2, M[2][n], fma(-hT1, M[1][n], hT0 * M[0][n])));
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const double x = M[e][pidx(c, a)], y = M[e][pidx(c, b)];
        s = ((e == 0) != (c == 0)) ? fma(-x, y, s) : fma(x, y, s);
      }
    S[n] = s;
  }
  // twice the lowered Christoffels, in place: G_a[bc] = D_b[ac] + D_c[ab] - D_a[bc]
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = a + 1; b < 4; ++b) {
#pragma unroll
      for (int c = b + 1; c < 4; ++c) {
        double &x = M[a][pidx(b, c)], &y = M[b][pidx(a, c)], &z = M[c][pidx(a, b)];
        const double t = x + y + z;
        x = fma(-2.0, x, t);
        y = fma(-2.0, y, t);
        z = fma(-2.0, z, t);
      }
      {
        double &p = M[a][pidx(b, b)], &q = M[b][pidx(a, b)];  // G_a[bb], G_b[ab]
        const double t = p;
        p = fma(2.0, q, -p);
        q = t;
      }
      {
        double &p = M[b][pidx(a, a)], &q = M[a][pidx(a, b)];  // G_b[aa], G_a[ab]
        const double t = p;
        p = fma(2.0, q, -p);
        q = t;
      }
    }
  const double hH0 = 0.5 * H[0], hH1 = 0.5 * H[1], hH2 = 0.5 * H[2], hH3 = 0.5 * H[3];
#pragma unroll
  for (int n = 0; n < NC; ++n) {
    const int a = prow(n), b = pcol(n);
    double d = M[a][0] * M[b][0], o = 0.0;
    d = fma(M[a][4], M[b][4], d);
    d = fma(M[a][7], M[b][7], d);
    d = fma(M[a][9], M[b][9], d);
    o = M[a][5] * M[b][5];
    o = fma(M[a][6], M[b][6], o);
    o = fma(M[a][8], M[b][8], o);
    o = fma(-M[a][1], M[b][1], o);
    o = fma(-M[a][2], M[b][2], o);
    o = fma(-M[a][3], M[b][3], o);
    d = fma(2.0, o, d);
    double s = fma(-0.25, d, S[n]);
    s = fma(-hH0, M[0][n], s);
    s = fma(hH1, M[1][n], s);
    s = fma(hH2, M[2][n], s);
    S[n] = fma(hH3, M[3][n], s);
  }
  // the damping (t_n = -1, t^c C_c = C_n)
  const double hg = 0.5 * g0, k1 = (1.0 + g2) * C0;
  S[0] = fma(hg, fma(-2.0, C0, k1), S[0]);
  S[1] = fma(-hg, C1, S[1]);
  S[2] = fma(-hg, C2, S[2]);
  S[3] = fma(-hg, C3, S[3]);
  S[4] = fma(-hg, k1, S[4]);
  S[7] = fma(-hg, k1, S[7]);
  S[9] = fma(-hg, k1, S[9]);
}

// The stage epilogue's arrays and coefficients. Stages 1-4 are RhsArgs's
// accumulator recurrences; 11-14 keep the stage values instead of an
// accumulator (Y1 = u + dt/2 k1, Y2 = u + dt/2 k2, Y3 = u + dt k3):
//   11: Y1 = u + c k (u the stage input's own point)   12, 13: Y = u + c k
//   14: u' = u + ((Y1 - u) + 2 (Y2 - u) + (Y3 - u))/3 + dt/6 k (Y3 the stage input)
// which is RK4's u + dt (k1 + 2 k2 + 2 k3 + k4)/6. Per variable they read and
// write 13 values a step instead of 18, and round each of the three
// differences once (half an ulp of u each, over 3) where the accumulator
// rounds three times. Not where a limiter changes the stage values (range
// bounds, :pasted) or the fill projects them (mirrors).
// STAGE 0 stores k (the rhs! verb).
enum { STAGE_STORE = 0, STAGE_Y1 = 11, STAGE_Y2 = 12, STAGE_Y3 = 13, STAGE_Y4 = 14 };
struct StageIO {
  int stage;
  double cacc, cnext;
  const double* us;   // u_n (1-3, 12-14)
  double* usw;        // u_{n+1} (4)
  double* acc;        // the accumulator (1-4), or Y1 (14)
  const double* y2;   // Y2 (14)
  double* out;        // the next stage's input; k (0)
  int images;         // 11-14: out's images across the periodic faces too (stage_wraps)
};
// A point's images across the periodic faces; a mesh of at least 2 G points an
// axis has one an axis at most.
struct Images {
  int mask;  // per axis two bits: 1 the image lies above, 2 below
  int n[3];  // the axes' lengths in bytes
};
template <bool ON>
__device__ __forceinline__ Images images_of(const Brick& k, int on, int x, int y, int z) {
  Images m{0, {8 * k.n[0], 8 * (int)k.py * k.n[1], 8 * (int)k.pz * k.n[2]}};
  if constexpr (ON) {
    if (on) {
      const int p[3] = {x, y, z};
#pragma unroll
      for (int d = 0; d < 3; ++d) m.mask |= (p[d] < k.G ? 1 : p[d] >= k.n[d] - k.G ? 2 : 0) << (2 * d);
    }
  }
  return m;
}
// The epilogue's kinds, compiled apart so that a kind's loads are unconditional:
// loads under a branch make the wait for them a wait for every load in flight,
// the next component's prefetch among them.
enum { K_Y1, K_Y23, K_Y4, K_C1, K_C23, K_C4, K_STORE };
struct EpiIn {
  double u, a, b;
};
// A value at 32-bit byte offset o of a uniform base: kept as a scalar base and
// a lane offset (hidden from the optimiser, which would widen the offset
// outside a loop and add in 64 bits inside it).
__device__ __forceinline__ double lane_ld(const double* p, unsigned& o) {
  asm volatile("" : "+v"(o));
  return *(TGH_GLOBAL const double*)((TGH_GLOBAL const char*)p + o);
}
__device__ __forceinline__ void lane_st(double* p, unsigned& o, double x) {
  asm volatile("" : "+v"(o));
  *(TGH_GLOBAL double*)((TGH_GLOBAL char*)p + o) = x;
}
// Variable v of an array with field stride ss.
__device__ __forceinline__ double field_ld(const double* p, int v, long ss, unsigned& o) {
  return lane_ld(p + (long)v * ss, o);
}
__device__ __forceinline__ void field_st(double* p, int v, long ss, unsigned& o, double x) {
  lane_st(p + (long)v * ss, o, x);
}
template <int K>
__device__ __forceinline__ EpiIn stage_load(const StageIO& s, int v, long ss, unsigned& o) {
  EpiIn e{0.0, 0.0, 0.0};
  if (K == K_Y23 || K == K_Y4 || K == K_C1 || K == K_C23) e.u = field_ld(s.us, v, ss, o);
  if (K == K_Y4 || K == K_C23 || K == K_C4) e.a = field_ld(s.acc, v, ss, o);
  if (K == K_Y4) e.b = field_ld(s.y2, v, ss, o);
  return e;
}
template <int K, bool IMG>
__device__ __forceinline__ void stage_store(const StageIO& s, int v, long ss, unsigned& o, double own, const EpiIn& e,
                                            double k, const Images& im) {
#pragma clang fp contract(off)
  double x = k;
  if (K == K_Y1) x = fma(s.cnext, k, own);
  if (K == K_Y23 || K == K_C1 || K == K_C23) x = fma(s.cnext, k, e.u);
  if (K == K_Y4) x = e.u + fma(fma(2.0, e.b - e.u, (e.a - e.u) + (own - e.u)), 1.0 / 3.0, s.cacc * k);
  if (K == K_C1) field_st(s.acc, v, ss, o, fma(s.cacc, k, e.u));
  if (K == K_C23) field_st(s.acc, v, ss, o, fma(s.cacc, k, e.a));
  if (K == K_C4) {
    x = fma(s.cacc, k, e.a);
    field_st(s.usw, v, ss, o, x);
  }
  field_st(s.out, v, ss, o, x);
  if constexpr (IMG && (K == K_Y1 || K == K_Y23 || K == K_Y4)) {
    if (im.mask) {
#pragma unroll
      for (int m = 1; m < 8; ++m) {
        unsigned oi = o;
        bool has = true;
#pragma unroll
        for (int d = 0; d < 3; ++d)
          if (m >> d & 1) {
            const int b = im.mask >> (2 * d) & 3;
            has = has && b;
            oi += (unsigned)(b == 1 ? im.n[d] : -im.n[d]);
          }
        if (has) field_st(s.out, v, ss, oi, x);
      }
    }
  }
}
template <int K>
struct KindC {
  static constexpr int value = K;
};

// The tile of a workgroup of 256 threads, one point a thread: 16 x 4 x 4 on
// the brick (a row of 16 doubles is a 128-byte line), 17 x 5 x 3 on a block of
// 17^3 owned points (80 % of the threads busy, where 16 x 4 x 4 would keep 43
// %): the octree of 2416 blocks takes 5.6 ms a stage where the two kernels it
// replaces took 6.2 + 4.1. The shape is the same for every N: away from 16 it
// keeps fewer threads busy (22 % at N = 6, 57 % at 12, 52 % at 20) and is still
// the faster. Steps of a three-level forest over one box with blocks of N = 6,
// 8, 10, 12, 16, 20, 24 and 32 take 77, 51, 40, 39, 37, 38, 37 and 45 ms, where
// the two kernels took 99, 74, 56, 55, 58, 52, 53 and 70.
enum { TILE_BRICK = 0, TILE_BLOCK = 1 };
template <int Q, int T> struct StageTile {
  static constexpr int X = T == TILE_BRICK ? 16 : 17, Y = T == TILE_BRICK ? 4 : 5, Z = T == TILE_BRICK ? 4 : 3;
  static constexpr int NP = X * Y * Z;       // points
  static constexpr int R = W<Q>::R, H = R + 1;
  // h's box (halo R: first, second and mixed derivatives)
  static constexpr int BX = X + 2 * R, BY = Y + 2 * R, BZ = Z + 2 * R, BV = BX * BY * BZ;
  // Pi on the three axis lines (halo H: first derivatives and dissipation), an array an axis
  static constexpr int PX = (X + 2 * H) * Y * Z, PY = X * (Y + 2 * H) * Z, PZ = X * Y * (Z + 2 * H);
  static constexpr int LV = BV + PX + PY + PZ;
  // two buffers where two workgroups' fit a CU's 160 KB beside the coefficients
  static constexpr int NB = (2 * LV + NC * 256) * 8 <= 80 * 1024 ? 2 : 1;
  static constexpr int NH = (BV + 255) / 256;                         // h loads a thread
  static constexpr int HX = 2 * H * Y * Z, HY = X * 2 * H * Z, HZ = X * Y * 2 * H;
  static constexpr int NHALO = HX + HY + HZ, NPL = (NHALO + 255) / 256;  // Pi halo loads a thread
};

// f(KindC<K>) of the stage's kind: the stage-value kinds on the brick, the
// accumulator's there where a limiter asks for it and on blocks.
template <int T, class F>
__device__ __forceinline__ void stage_kind(int stage, const F& f) {
  if constexpr (T == TILE_BRICK) {
    if (stage == STAGE_Y1) return f(KindC<K_Y1>{});
    if (stage == STAGE_Y2 || stage == STAGE_Y3) return f(KindC<K_Y23>{});
    if (stage == STAGE_Y4) return f(KindC<K_Y4>{});
  } else {
    if (stage == STAGE_STORE) return f(KindC<K_STORE>{});
  }
  if (stage == 1) return f(KindC<K_C1>{});
  if (stage < 4) return f(KindC<K_C23>{});
  return f(KindC<K_C4>{});
}

// One tile, corner (X0, Y0, Z0), of the stage's right-hand side: the head with
// h's results (where vb is 0), and the Pi components vb to ve - 1.
template <int Q, int GAUGE, int HOLE, int T>
__device__ __forceinline__ void stage_tile(const RhsArgs& a, const Brick& k, const double* __restrict__ W,
                                           const double* __restrict__ Hsrc, const StageIO& io, bool state_out,
                                           int X0, int Y0, int Z0, int vb = 0, int ve = NC) {
#pragma clang fp contract(off)
  using TT = StageTile<Q, T>;
  constexpr int TX = TT::X, TY = TT::Y, TZ = TT::Z, R = TT::R, H = TT::H;
  __shared__ double sh[TT::NB * TT::LV];
  __shared__ double sc1[NC * 256];
  const int t = threadIdx.x;
  const int tp = t < TT::NP ? t : 0;
  const int lx = tp % TX, ly = (tp / TX) % TY, lz = tp / (TX * TY);
  const int x = X0 + lx, y = Y0 + ly, z = Z0 + lz;
  const bool valid = t < TT::NP && x < k.n[0] && y < k.n[1] && z < k.n[2];
  const CaseP& c = a.c;
  const int py = (int)k.py, pz = (int)k.pz;
  // a thread without a point reads the tile's first one
  const int ioff = k.XO + py * k.G + pz * k.G;  // brick_index in 32 bits: x + py y + pz z + ioff
  const int off = valid ? x + py * y + pz * z + ioff : X0 + py * Y0 + pz * Z0 + ioff;
  unsigned so = (unsigned)off * 8u;  // where the outputs go, in bytes, and their field stride
  long ss = k.fs;
  if (T == TILE_BLOCK && state_out) {
    const int P = a.g.P;
    ss = (long)P * P * P;
    so = valid ? (unsigned)(x + P * (y + P * z)) * 8u : 0u;
  }
  constexpr bool IMG = HOLE == 0 && T == TILE_BRICK;
  const Images im = images_of<IMG>(k, io.images, x, y, z);
  double* c1 = sc1 + t;
  double pb[3], pdivb = 0.0, pA[6], pw = 1.0, pe = 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i) pb[i] = 0.0;
#pragma unroll
  for (int i = 0; i < 6; ++i) pA[i] = 0.0;
  const double ih = k.inv_h;
  auto at = [&](int v, int o) -> double {  // variable v at element offset o of the array: 32-bit lane offsets
    const char* base = (const char*)(W + (long)v * k.fs);
    return *(const double*)(base + (unsigned)o * 8u);
  };

  // ---- the head ----
  if (valid) {
    const double xp[3] = {grid_coord(k.lo[0], x + k.gx0[0], k.h), grid_coord(k.lo[1], y + k.gx0[1], k.h),
                          grid_coord(k.lo[2], z + k.gx0[2], k.h)};
    long lslot = 0;
    if (HOLE && a.lbox)
      lslot = layer_slot((x + k.gx0[0]) << k.lsh, (y + k.gx0[1]) << k.lsh, (z + k.gx0[2]) << k.lsh, a.lB);
    double r;
    if (frozen_core<HOLE>(c, a.t, xp, r)) {
      double dh[NC], dP[NC];
      const GlobalSrc src{W + off, k.fs, py, pz};
      core_rates<GAUGE, HOLE>(a, xp, lslot, src, dh, dP);
      if (vb == 0)
        stage_kind<T>(io.stage, [&](auto kc) {
          constexpr int K = decltype(kc)::value;
#pragma unroll
          for (int v = 0; v < NC; ++v)
            stage_store<K, IMG>(io, v, ss, so, at(v, off), stage_load<K>(io, v, ss, so), dh[v], im);
        });
#pragma unroll
      for (int v = 0; v < NC; ++v) c1[v * 256] = dP[v];
      pw = -1.0;
    } else {
      double h[NC], M[4][NC], P[NC];
      {
        double w1[R + 1];
#pragma unroll
        for (int q = 1; q <= R; ++q) w1[q] = ih * ::tgh::W<Q>::d1[R + q];
        // the loads of the variable DEPTH ahead are in flight while one is differenced
        constexpr int DEPTH = Q <= 4 ? 2 : 1, NB = DEPTH + 1;
        double raw[NB][3][2 * H + 1];
        auto load = [&](int v) {
          double(*b)[2 * H + 1] = raw[v % NB];
          b[0][H] = at(v, off);
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const int st = d == 0 ? 1 : d == 1 ? py : pz;
#pragma unroll
            for (int q = 1; q <= H; ++q) {
              b[d][H + q] = at(v, off + q * st);
              b[d][H - q] = at(v, off - q * st);
            }
          }
        };
#pragma unroll
        for (int v = 0; v < DEPTH; ++v) load(v);
#pragma unroll
        for (int v = 0; v < NC; ++v) {
          if (v + DEPTH < NC) load(v + DEPTH);
          if (v == NC - 1) {
#pragma unroll
            for (int q = 0; q < NC; ++q) P[q] = at(NC + q, off);
          }
          __builtin_amdgcn_sched_barrier(0);
          const double(*b)[2 * H + 1] = raw[v % NB];
          h[v] = b[0][H];
          double ks[H + 1];
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            double g = 0.0;
#pragma unroll
            for (int q = 1; q <= H; ++q) {
              const double p = b[d][H + q], m = b[d][H - q];
              if (q <= R) g = q == 1 ? w1[1] * (p - m) : fma(w1[q], p - m, g);
              ks[q] = d == 0 ? p + m : ks[q] + (p + m);
            }
            M[1 + d][v] = g;
          }
          double ko = (3.0 * ::tgh::W<Q>::ko[H]) * h[v];
#pragma unroll
          for (int q = 1; q <= H; ++q) ko = fma(::tgh::W<Q>::ko[H + q], ks[q], ko);
          M[0][v] = ko;
          // formed here: moved past the branches below, the sums would keep
          // their nineteen inputs alive
#pragma unroll
          for (int d = 0; d < 4; ++d) asm volatile("" : "+v"(M[d][v]));
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      Frame f;
      make_frame(h, f);
      const double r2 = radius2(c, a.t, xp);
      pe = dissipation_stage(c, r2) * ih;
      double wgt = 1.0, rho = 0.0;
      const bool layer = HOLE && r < c.r1;
      if (layer) {
        const double sl = (r - c.r0) / (c.r1 - c.r0);
        wgt = smoothstep_stage(sl / c.w_ramp);
        rho = c.interior == INT_FROZEN ? 0.0 : c.rho_max * smoothstep_stage((1.0 - sl) / c.rho_ramp);
      }
      constexpr bool MOVE = (bg_set_for(GAUGE) & BGS_MOVING) != 0;
      const bool follows = MOVE && c.moving && c.interior == INT_DAMPED;
      const double om = 1.0 - wgt;
      const double* lb = HOLE ? a.lbox + lslot : nullptr;
      // D_n h = Pi / sqrt(gamma) + KO / alpha, d_t h = beta^i d_i h + alpha D_n h
      const double ek = c.has_diss ? pe * f.ra : 0.0;
      double dt4[4], dth[NC];
#pragma unroll
      for (int v = 0; v < NC; ++v) {
        const double dn = fma(P[v], f.isg, ek * M[0][v]);
        M[0][v] = dn;
        double d = fma(f.bu[0], M[1][v], fma(f.bu[1], M[2][v], fma(f.bu[2], M[3][v], f.al * dn)));
        if (v < 4) dt4[v] = d;
        if (HOLE && layer) {
          const double ue = lb[v * a.lB3];
          d = fma(wgt, d, -(rho * (h[v] - ue)));
          if (follows) d = fma(om, lb[(2 * NC + v) * a.lB3], d);
        }
        dth[v] = d;
      }
      if (vb == 0)
        stage_kind<T>(io.stage, [&](auto kc) {
          constexpr int K = decltype(kc)::value;
#pragma unroll
          for (int v0 = 0; v0 < NC; v0 += 5) {
            EpiIn e[5];
#pragma unroll
            for (int q = 0; q < 5; ++q) e[q] = stage_load<K>(io, v0 + q, ss, so);
#pragma unroll
            for (int q = 0; q < 5; ++q) stage_store<K, IMG>(io, v0 + q, ss, so, h[v0 + q], e[q], dth[v0 + q], im);
          }
        });
      // the gauge source in the frame, and its symmetrised derivative dHs
      double Hf[4] = {0.0, 0.0, 0.0, 0.0}, dHs[NC];
      constexpr bool HAS_H = gauge_has_source(GAUGE);
      if constexpr (HAS_H) {
        double Hl[4];
        if constexpr (GAUGE == GAUGE_SAMPLED) {
          // brick fields on the brick, the state's layout on a block
          const long P1 = a.g.P, hs = T == TILE_BRICK ? k.fs : P1 * P1 * P1;
          const double* Hp = Hsrc + (T == TILE_BRICK ? (long)off : x + P1 * (y + P1 * z));
#pragma unroll
          for (int q = 0; q < 4; ++q) Hl[q] = Hp[q * hs];
#pragma unroll
          for (int n = 0; n < NC; ++n)  // dH[c][a] at field 4 + c + 4 a
            dHs[n] = Hp[(4 + prow(n) + 4 * pcol(n)) * hs] + Hp[(4 + pcol(n) + 4 * prow(n)) * hs];
        } else {
          // H_a = q w_a, q = -K / Dn: d_c H_a = q d_c w_a + w_a d_c q (KerrSchildSource)
          double w[4], K, sw;
          if constexpr (GAUGE == GAUGE_KS) {
#pragma unroll
            for (int q = 0; q < 4; ++q) w[q] = h[q];
            K = w[0];
            sw = c.bg.a * w[3];
          } else {
            const double* u = c.ks_u;
#pragma unroll
            for (int q = 0; q < 4; ++q)
              w[q] = fma(h[pidx(q, 0)], u[0], dot3(h[pidx(q, 1)], u[1], h[pidx(q, 2)], u[2], h[pidx(q, 3)], u[3]));
            K = fma(u[0], w[0], dot3(u[1], w[1], u[2], w[2], u[3], w[3]));
            sw = fma(c.ks_S[0], w[0], dot3(c.ks_S[1], w[1], c.ks_S[2], w[2], c.ks_S[3], w[3]));
          }
          const double Ms = c.bg.M, rad = fma(-sw, sw, Ms * Ms);
          const double root = rad > 0.0 ? sqrt(rad) : 0.0;
          const double iD = 1.0 / (Ms + root);
          const double q = -K * iD;
          // d_c q = -iD d_c K + K iD^2 d_c Dn, d_c Dn = -sw d_c(sw) / root
          const double k3 = root > 0.0 ? q * iD * sw / root : 0.0;
          double dw[4][4], dq[4];
          if constexpr (GAUGE == GAUGE_KS) {
#pragma unroll
            for (int a2 = 0; a2 < 4; ++a2) {
              dw[0][a2] = dt4[a2];
#pragma unroll
              for (int d = 1; d < 4; ++d) dw[d][a2] = M[d][a2];
            }
            const double k3a = k3 * c.bg.a;
#pragma unroll
            for (int d = 0; d < 4; ++d) dq[d] = fma(k3a, dw[d][3], -(iD * dw[d][0]));
          } else {
            const double* u = c.ks_u;
#pragma unroll
            for (int d = 0; d < 4; ++d) {
              double D[NC];
#pragma unroll
              for (int v = 0; v < NC; ++v)
                D[v] = d > 0 ? M[d][v]
                             : fma(f.bu[0], M[1][v], fma(f.bu[1], M[2][v], fma(f.bu[2], M[3][v], f.al * M[0][v])));
#pragma unroll
              for (int a2 = 0; a2 < 4; ++a2)
                dw[d][a2] = fma(D[pidx(a2, 0)], u[0],
                                fma(D[pidx(a2, 1)], u[1], fma(D[pidx(a2, 2)], u[2], D[pidx(a2, 3)] * u[3])));
              const double dK =
                  fma(u[0], dw[d][0], fma(u[1], dw[d][1], fma(u[2], dw[d][2], u[3] * dw[d][3])));
              const double dS = fma(c.ks_S[0], dw[d][0],
                                    fma(c.ks_S[1], dw[d][1], fma(c.ks_S[2], dw[d][2], c.ks_S[3] * dw[d][3])));
              dq[d] = fma(k3, dS, -(iD * dK));
            }
          }
#pragma unroll
          for (int n = 0; n < NC; ++n) {
            const int i = prow(n), j = pcol(n);
            dHs[n] = fma(q, dw[i][j] + dw[j][i], fma(dq[i], w[j], dq[j] * w[i]));
          }
#pragma unroll
          for (int s = 0; s < 4; ++s) Hl[s] = q * w[s];
        }
        Hf[0] = (Hl[0] - dot3(f.bu[0], Hl[1], f.bu[1], Hl[2], f.bu[2], Hl[3])) * f.ra;
        Hf[1] = f.e11 * Hl[1];
        Hf[2] = dot2(f.e21, Hl[1], f.e22, Hl[2]);
        Hf[3] = dot3(f.e31, Hl[1], f.e32, Hl[2], f.e33, Hl[3]);
      }
      // the derivatives into the frame: the derivative's own index, then the tensor's
#pragma unroll
      for (int v = 0; v < NC; ++v) {
        const double d1 = M[1][v], d2 = M[2][v], d3 = M[3][v];
        M[1][v] = f.e11 * d1;
        M[2][v] = dot2(f.e21, d1, f.e22, d2);
        M[3][v] = dot3(f.e31, d1, f.e32, d2, f.e33, d3);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) to_frame(f, M[e]);
      // the fluxes' divergences (metric_divergences): d_i beta^i = alpha sum_A D_A g_nA,
      // d_i (alpha sqrt(gamma) gamma^ij) = alpha sqrt(gamma) e_Aj w_A with
      // w_A = (D_A ln(alpha sqrt gamma)) - sum_B D_B g_AB; its product with d_j h
      // is a sum of the same D_A h the source contracts, and is formed there
      pdivb = f.al * (M[1][1] + M[2][2] + M[3][3]);
      double wA[3];
#pragma unroll
      for (int A = 0; A < 3; ++A) {
        const double* m = M[1 + A];
        wA[A] = fma(0.5, (m[4] + m[7] + m[9]) - m[0],
                    -(M[1][pidx(1, 1 + A)] + M[2][pidx(2, 1 + A)] + M[3][pidx(3, 1 + A)]));
      }
      const double g0 = damping_stage(c, r2);
      double S[NC];
      frame_source(M, Hf, wA, g0, c.g2, S);
      from_frame(f, S);
      const double as = f.al * f.sg, m2as = -2.0 * as;
#pragma unroll
      for (int v = 0; v < NC; ++v) {
        double s = m2as * S[v];
        if constexpr (HAS_H) s = fma(as, dHs[v], s);
        if (HOLE && layer) {
          const double ue = lb[(NC + v) * a.lB3];
          s = fma(wgt, s, -(rho * (at(NC + v, off) - ue)));
          if (follows)
            s = fma(om, (lb[(3 * NC + v) * a.lB3] - lb[(4 * NC + v) * a.lB3]) / ((a.t + c.delta) - (a.t - c.delta)), s);
        }
        c1[v * 256] = s;
      }
      if (HOLE && layer) pw = wgt;
      // the Pi components' coefficients, scaled by the spacings of their stencils
      const double as2 = as * ih * ih;
      pb[0] = ih * f.bu[0];
      pb[1] = ih * f.bu[1];
      pb[2] = ih * f.bu[2];
      pA[0] = as2 * dot3(f.e11, f.e11, f.e21, f.e21, f.e31, f.e31);
      pA[1] = 2.0 * as2 * dot2(f.e21, f.e22, f.e31, f.e32);
      pA[2] = 2.0 * as2 * (f.e31 * f.e33);
      pA[3] = as2 * dot2(f.e22, f.e22, f.e32, f.e32);
      pA[4] = 2.0 * as2 * (f.e32 * f.e33);
      pA[5] = as2 * (f.e33 * f.e33);
    }
  }
  if (!c.has_diss) pe = 0.0;

  // ---- the ten Pi components ----
  // Each component's h and Pi go through registers into LDS, the next one's
  // loads in flight while the present one is computed.
  const int xm = k.n[0] + k.G - 1, ym = k.n[1] + k.G - 1, zm = k.n[2] + k.G - 1;  // the stored extent
  auto elem = [&](int ex, int ey, int ez) -> unsigned {  // its byte offset in a field
    return (unsigned)(min(ex, xm) + py * min(ey, ym) + pz * min(ez, zm) + ioff) * 8u;
  };
  unsigned go[TT::NH], gp[TT::NPL];
  int lp[TT::NPL];
#pragma unroll
  for (int j = 0; j < TT::NH; ++j) {
    const int i = min(t + 256 * j, TT::BV - 1);
    go[j] = elem(X0 - R + i % TT::BX, Y0 - R + (i / TT::BX) % TT::BY, Z0 - R + i / (TT::BX * TT::BY));
  }
#pragma unroll
  for (int j = 0; j < TT::NPL; ++j) {
    int i = min(t + 256 * j, TT::NHALO - 1);
    int ex, ey, ez;
    if (i < TT::HX) {
      const int q = i % (2 * H), row = i / (2 * H);
      ex = q < H ? q - H : TX + q - H;
      ey = row % TY;
      ez = row / TY;
      lp[j] = row * (TX + 2 * H) + ex + H;
    } else if (i < TT::HX + TT::HY) {
      i -= TT::HX;
      const int q = (i / TX) % (2 * H);
      ex = i % TX;
      ez = i / (TX * 2 * H);
      ey = q < H ? q - H : TY + q - H;
      lp[j] = TT::PX + (ez * (TY + 2 * H) + ey + H) * TX + ex;
    } else {
      i -= TT::HX + TT::HY;
      const int q = i / (TX * TY);
      ex = i % TX;
      ey = (i / TX) % TY;
      ez = q < H ? q - H : TZ + q - H;
      lp[j] = TT::PX + TT::PY + ((ez + H) * TY + ey) * TX + ex;
    }
    gp[j] = elem(X0 + ex, Y0 + ey, Z0 + ez);
  }
  unsigned offc = elem(x, y, z);
  double rh[TT::NH], rp[TT::NPL], rc;
  auto fetch = [&](int v) {
    const double *wh = W + (long)v * k.fs, *wp = W + (long)(NC + v) * k.fs;
#pragma unroll
    for (int j = 0; j < TT::NH; ++j) rh[j] = lane_ld(wh, go[j]);
#pragma unroll
    for (int j = 0; j < TT::NPL; ++j) rp[j] = lane_ld(wp, gp[j]);
    rc = lane_ld(wp, offc);
  };
  fetch(vb);
  const int ch = (lx + R) + TT::BX * ((ly + R) + TT::BY * (lz + R));
  const int cpx = (ly + TY * lz) * (TX + 2 * H) + lx + H;
  const int cpy = TT::PX + (lz * (TY + 2 * H) + ly + H) * TX + lx;
  const int cpz = TT::PX + TT::PY + ((lz + H) * TY + ly) * TX + lx;
  stage_kind<T>(io.stage, [&](auto kc) {
    constexpr int K = decltype(kc)::value;
#pragma unroll 1
    for (int v = vb; v < ve; ++v) {
      double* bh = sh + (TT::NB == 2 ? (v & 1) * TT::LV : 0);
      double* bp = bh + TT::BV;
      if (TT::NB == 1) __syncthreads();  // the previous component's reads are done
#pragma unroll
      for (int j = 0; j < TT::NH; ++j)
        if (t + 256 * j < TT::BV) bh[t + 256 * j] = rh[j];
#pragma unroll
      for (int j = 0; j < TT::NPL; ++j)
        if (t + 256 * j < TT::NHALO) bp[lp[j]] = rp[j];
      const double P = rc;
      if (t < TT::NP) {
        bp[cpx] = rc;
        bp[cpy] = rc;
        bp[cpz] = rc;
      }
      // with two buffers this barrier also separates the reads of the buffer two
      // components back from the writes above
      __syncthreads();
      const EpiIn e = stage_load<K>(io, NC + v, ss, so);
      if (v + 1 < ve) fetch(v + 1);
      const double* ph = bh + ch;
      constexpr int st[3] = {1, TT::BX, TT::BX * TT::BY};
      constexpr int pst[3] = {1, TX, TX * TY};
      const int pc0[3] = {cpx, cpy, cpz};
      double hl[3][2 * R], pl[3][2 * H], mx[2][4 * R * R];
      const double hc = ph[0];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
#pragma unroll
        for (int q = 1; q <= R; ++q) {
          hl[d][2 * q - 2] = ph[q * st[d]];
          hl[d][2 * q - 1] = ph[-q * st[d]];
        }
      }
      auto lines = [&]() {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const double* pp = bp + pc0[d];
#pragma unroll
          for (int q = 1; q <= H; ++q) {
            pl[d][2 * q - 2] = pp[q * pst[d]];
            pl[d][2 * q - 1] = pp[-q * pst[d]];
          }
        }
      };
      auto mixed = [&](int m, double* o) {
        const int s1 = m == 2 ? st[1] : 1, s2 = m == 0 ? st[1] : st[2];
        int n = 0;
#pragma unroll
        for (int q1 = 1; q1 <= R; ++q1)
#pragma unroll
          for (int q2 = 1; q2 <= R; ++q2) {
            o[n++] = ph[q1 * s1 + q2 * s2];
            o[n++] = ph[q1 * s1 - q2 * s2];
            o[n++] = ph[-q1 * s1 + q2 * s2];
            o[n++] = ph[-q1 * s1 - q2 * s2];
          }
      };
      // products of the first-derivative weights over the differences of
      // opposite corners
      auto mixed_sum = [&](const double* o) {
        double g = 0.0;
        int n = 0;
#pragma unroll
        for (int q1 = 1; q1 <= R; ++q1)
#pragma unroll
          for (int q2 = 1; q2 <= R; ++q2) {
            const double w = ::tgh::W<Q>::d1[R + q1] * ::tgh::W<Q>::d1[R + q2];
            const double d = (o[n] - o[n + 1]) - (o[n + 2] - o[n + 3]);
            g = n == 0 ? w * d : fma(w, d, g);
            n += 4;
          }
        return g;
      };
      lines();
      mixed(0, mx[0]);
      double s = pdivb * P, ks[H + 1];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        double g2 = ::tgh::W<Q>::d2[R] * hc;
#pragma unroll
        for (int q = 1; q <= R; ++q) g2 = fma(::tgh::W<Q>::d2[R + q], hl[d][2 * q - 2] + hl[d][2 * q - 1], g2);
        s = fma(pA[d == 0 ? 0 : d == 1 ? 3 : 5], g2, s);
        double gP = 0.0;
#pragma unroll
        for (int q = 1; q <= H; ++q) {
          const double p = pl[d][2 * q - 2], m = pl[d][2 * q - 1];
          if (q <= R) gP = q == 1 ? ::tgh::W<Q>::d1[R + 1] * (p - m) : fma(::tgh::W<Q>::d1[R + q], p - m, gP);
          ks[q] = d == 0 ? p + m : ks[q] + (p + m);
        }
        s = fma(pb[d], gP, s);
      }
      double ko = (3.0 * ::tgh::W<Q>::ko[H]) * P;
#pragma unroll
      for (int q = 1; q <= H; ++q) ko = fma(::tgh::W<Q>::ko[H + q], ks[q], ko);
      s = fma(pe, ko, s);
      mixed(1, mx[1]);
      s = fma(pA[1], mixed_sum(mx[0]), s);
      mixed(2, mx[0]);
      s = fma(pA[2], mixed_sum(mx[1]), s);
      s = fma(pA[4], mixed_sum(mx[0]), s);
      // in the frozen core (pw < 0) the rate is the coefficient itself
      s = (pw < 0.0 ? 0.0 : s * pw) + c1[v * 256];
      if (valid) stage_store<K, IMG>(io, NC + v, ss, so, P, e, s, im);
    }
  });
}

template <int Q>
__host__ __device__ inline int brick_stage_tiles(const Brick& k) {
  using TT = StageTile<Q, TILE_BRICK>;
  return ((k.n[0] + TT::X - 1) / TT::X) * ((k.n[1] + TT::Y - 1) / TT::Y) * ((k.n[2] + TT::Z - 1) / TT::Z);
}
// How many workgroups share a tile's Pi components, each with the head of its
// own, on a mesh without an interior: as many as leave at most one workgroup a
// CU, where a tile takes as long as its instructions do one after another. A
// stage at q = 4 in 1, 2 and 5 parts: 16 tiles 31, 24 and 20 us; 72 tiles 32,
// 25 and 27; 128 tiles 33, 26 and 35; 243 tiles 34, 34 and 52.
__host__ __device__ inline int stage_parts(int tiles) { return tiles * 5 <= 256 ? 5 : tiles * 2 <= 256 ? 2 : 1; }
// The brick's tiles in launch order: the XCDs take contiguous ranges of slabs
// in y, each swept plane of tiles by plane of tiles in z, so that the eight
// sweep the same planes and share them in the memory-side cache (a step of
// 27.1 ms against 28.2 with the XCDs on slabs in z).
template <int Q>
__device__ __forceinline__ void stage_brick_tile(const Brick& k, int L, int& X0, int& Y0, int& Z0) {
  using TT = StageTile<Q, TILE_BRICK>;
  const int nx = (k.n[0] + TT::X - 1) / TT::X, ny = (k.n[1] + TT::Y - 1) / TT::Y, nz = (k.n[2] + TT::Z - 1) / TT::Z;
  const int gy = (ny + NUM_XCD - 1) / NUM_XCD;  // tiles of a slab
  const int per = nx * gy * nz;
  const int sl = L / per;
  int r = L - sl * per;
  const int wy = min(gy, ny - sl * gy);
  X0 = (r % nx) * TT::X;
  r /= nx;
  Y0 = (sl * gy + r % wy) * TT::Y;
  Z0 = (r / wy) * TT::Z;
}
#define TGH_STAGE_KERNEL __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
template <int Q, int GAUGE, int HOLE>
TGH_STAGE_KERNEL void k_brick_stage(RhsArgs a, Brick k, const double* __restrict__ W, const double* __restrict__ Hsrc,
                                    StageIO io, int total) {
  a.t = stage_time(a.t, a.clock, a.toff);
  const int L = wg_logical(total);
  if (L >= total) return;  // uniform over the workgroup
  int X0, Y0, Z0;
  stage_brick_tile<Q>(k, L, X0, Y0, Z0);
  if constexpr (HOLE != 0) {
    stage_tile<Q, GAUGE, HOLE, TILE_BRICK>(a, k, W, Hsrc, io, false, X0, Y0, Z0);
  } else {
    // part blockIdx.y of the Pi components (stage_parts)
    const int parts = gridDim.y, part = blockIdx.y;
    stage_tile<Q, GAUGE, HOLE, TILE_BRICK>(a, k, W, Hsrc, io, false, X0, Y0, Z0, NC * part / parts,
                                           NC * (part + 1) / parts);
  }
}

// The block layout: tile wx of block b, each block's work array a brick. The
// stage's arrays in the work layout, or k into the state's layout.
__host__ __device__ inline int block_tiles(int P) {
  using TT = StageTile<4, TILE_BLOCK>;  // the same shape at every order
  return ((P + TT::X - 1) / TT::X) * ((P + TT::Y - 1) / TT::Y) * ((P + TT::Z - 1) / TT::Z);
}
template <int Q, int GAUGE, int HOLE>
__device__ __forceinline__ void stage_block(const RhsArgs& a, const double* __restrict__ W,
                                            const double* __restrict__ Hsrc, StageIO io, int lLmax, int b, int wx) {
  using TT = StageTile<Q, TILE_BLOCK>;
  const int P = a.g.P;
  const int tx = (P + TT::X - 1) / TT::X, ty = (P + TT::Y - 1) / TT::Y;
  const int X0 = (wx % tx) * TT::X, Y0 = ((wx / tx) % ty) * TT::Y, Z0 = (wx / (tx * ty)) * TT::Z;
  const Brick k = block_brick(a.g, b, lLmax);
  const long wb = (long)b * 20 * k.fs, sb = (long)b * 20 * P * P * P;
  const bool state_out = io.stage == STAGE_STORE;
  io.us += wb;
  io.usw += wb;
  io.acc += wb;
  io.out += state_out ? sb : wb;
  stage_tile<Q, GAUGE, HOLE, TILE_BLOCK>(a, k, W + wb, Hsrc ? Hsrc + sb : nullptr, io, state_out, X0, Y0, Z0);
}
template <int Q, int GAUGE, int HOLE>
TGH_STAGE_KERNEL void k_block_stage(RhsArgs a, const double* __restrict__ W, const double* __restrict__ Hsrc,
                                    StageIO io, int lLmax) {
  a.t = stage_time(a.t, a.clock, a.toff);
  int b, wx;
  if (!wg_map(block_tiles(a.g.P), a.g.nblocks, b, wx)) return;  // uniform over the workgroup
  stage_block<Q, GAUGE, HOLE>(a, W, Hsrc, io, lLmax, b, wx);
}

// Several problems in one launch (BatchEntry's table): each entry's tiles a
// range of logical workgroups from wg0.
__device__ __forceinline__ StageIO batch_io(const BatchEntry& e) {
  return StageIO{e.a.stage, e.a.cacc, e.a.cnext, (double*)e.us, (double*)e.us, (double*)e.acc, (double*)e.y2,
                 (double*)e.Wn, 0};
}
template <int Q, int GAUGE, int HOLE>
TGH_STAGE_KERNEL void k_brick_stage_batch(const BatchEntry* __restrict__ tab, int n, int total) {
  const int L = wg_logical(total);
  if (L >= total) return;  // uniform over the workgroup
  const BatchEntry& e = tab[batch_find(tab, n, L)];
  int X0, Y0, Z0;
  stage_brick_tile<Q>(e.k, L - e.wg0, X0, Y0, Z0);
  stage_tile<Q, GAUGE, HOLE, TILE_BRICK>(e.a, e.k, (const double*)e.W, (const double*)e.Hsrc, batch_io(e), false, X0,
                                         Y0, Z0);
}
template <int Q, int GAUGE, int HOLE>
TGH_STAGE_KERNEL void k_block_stage_batch(const BatchEntry* __restrict__ tab, int n, int total) {
  const int L = wg_logical(total);
  if (L >= total) return;  // uniform over the workgroup
  const BatchEntry& e = tab[batch_find(tab, n, L)];
  const int nt = block_tiles(e.a.g.P), loc = L - e.wg0, b = loc / nt;
  stage_block<Q, GAUGE, HOLE>(e.a, (const double*)e.W, (const double*)e.Hsrc, batch_io(e), e.lLmax, b, loc - b * nt);
}

}  // namespace tgh
