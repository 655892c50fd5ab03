// vfg_umodal.h -- the damaged-elasticity element in moment form.
//
// On one Q1 element (xi, eta, zeta in [-1,1]) every displacement derivative is
// a polynomial in the two other variables, d_x u = sum u_bc eta^b zeta^c with
// b, c in {0,1}, and the degradation s = v^2 + eta is at most quadratic in each
// variable.  The integrand s sigma : eps(w) has degree 4 per variable, which
// the reference's 3-point Gauss rule integrates exactly, so the element matrix
// depends on v only through the moments
//   M_pqr = <s xi^p eta^q zeta^r>,  p, q, r <= 2,
// of which the 23 with no more than two of the exponents at 2 and the rest
// matching a product of two derivatives occur.  A product of the element
// matrix then takes 21 4 x 4 blocks of moments (336 FMAs) instead of 27 Gauss
// points with nine stress entries each: 686 FP64 instructions per element
// against 1390.  The moments themselves are Simpson sums of s over the
// 3 x 3 x 3 points {-1, 0, 1} (z in closed form), where v needs additions only.
//
// Scaling: a pair of derivatives d, e carries hx^2 / (h_d h_e) (and its Lame
// ratio) as one constant, rounded once; kap = vol mu / (16 hx^2) times the
// constants of the moment sums.
#pragma once
#include "vfg_modal.h"

namespace vfg {

// launch constants of the element in moment form
template <typename T>
struct UModal {
  T kap;         // vol mu1 / (2304 hx^2): 1/16 (derivatives) x 1/4 (v sums) x 1/36 (Simpson in x and y); unit: / 16
  T eta4;        // 4 eta
  // hx^2 / (h_d h_e) times 1 (kx), lam / mu (kl), and for d = e lam / mu + 2 (k2)
  T kx[3][3], kl[3][3], k2[3];
  int cubic;     // all of kx are 1: the products by them are left out, with the same results
};
template <typename T>
inline UModal<T> make_umodal(const Grid &G, double lam1, double mu1, double eta, bool unit) {
  UModal<T> m;
  // formed in extended precision: each constant is rounded once
  const long double h[3] = {G.hx, G.hy, G.hz}, lr = (long double)lam1 / mu1;
  m.kap = T(h[1] * h[2] / h[0] * mu1 / (unit ? 16. : 2304.));
  m.eta4 = T(4. * eta);
  for (int d = 0; d < 3; d++) {
    for (int e = 0; e < 3; e++) {
      m.kx[d][e] = T(h[0] * h[0] / (h[d] * h[e]));
      m.kl[d][e] = T(lr * h[0] * h[0] / (h[d] * h[e]));
    }
    m.k2[d] = T((lr + 2) * h[0] * h[0] / (h[d] * h[d]));
  }
  m.cubic = 1;
  for (int d = 0; d < 3; d++) {
    for (int e = 0; e < 3; e++)
      if (m.kx[d][e] != T(1) || m.kl[d][e] != m.kl[0][0]) m.cubic = 0;
    if (m.k2[d] != m.k2[0]) m.cubic = 0;
  }
  return m;
}

// One face (node plane) of an element column, per displacement component: the
// value at the first corner, and of the differences to it the sum s, the x- and
// y-slope sums x, y and the twist w.  Derivatives are formed
// from nodal differences, not from sums of values, so a smooth field loses no
// digits to its mean.
template <typename T>
struct UFace {
  T a[3], s[3], x[3], y[3], w[3];
};
template <typename T>
__device__ __forceinline__ void uface_set(UFace<T> &F, int c, T x0, T x1, T x2, T x3) {
  const T b = x1 - x0, e = x2 - x0, d = x3 - x0;
  const T t = d - e;
  F.a[c] = x0;
  F.x[c] = t + b;                // (x1 + x3) - (x0 + x2)
  F.w[c] = t - b;                // (x0 + x3) - (x1 + x2)
  F.y[c] = T(2) * d - F.x[c];    // (x2 + x3) - (x0 + x1)
  F.s[c] = T(2) * d - F.w[c];    // x1 + x2 + x3 - 3 x0
}

// exponent of variable e in (modal i without d) * (modal j without dp)
constexpr int um_exp(int i, int d, int j, int dp, int e) {
  return (e == d ? 0 : um_pow(i, e)) + (e == dp ? 0 : um_pow(j, e));
}

// the moments of s = v^2 + eta times E, M[p][q][r], from v at the corners of the
// bottom (vb) and top (vt) faces; Ek = E kap.  A point between two corners
// holds their sum (v twice, s four times), the face centre the sum of four, so
// Simpson's middle weight 4 is already in the value.
template <typename T>
__device__ __forceinline__ void um_moments(const T *vb, const T *vt, T Ek, T eta4, T (&M)[3][3][3]) {
  T p[3][3], q[3][3];  // [y][x] at {-1, 0, 1}: v = (p + q zeta) / 2 at a corner column
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int i = 0; i < 2; i++) {
      p[2 * j][2 * i] = vb[j * 2 + i] + vt[j * 2 + i];
      q[2 * j][2 * i] = vt[j * 2 + i] - vb[j * 2 + i];
    }
#pragma unroll
  for (int j = 0; j < 3; j += 2) {
    p[j][1] = p[j][0] + p[j][2];
    q[j][1] = q[j][0] + q[j][2];
  }
#pragma unroll
  for (int i = 0; i < 3; i++) {
    p[1][i] = p[0][i] + p[2][i];
    q[1][i] = q[0][i] + q[2][i];
  }
  const T eta16 = T(4) * eta4, eta64 = T(16) * eta4;
  T zx[3][3][3];  // [r][q][x]: zeta- and eta-moments per x point
#pragma unroll
  for (int i = 0; i < 3; i++) {
    T z[3][3];  // [r][y], up to 1, 2/3, 1/3
#pragma unroll
    for (int j = 0; j < 3; j++) {
      const int mid = (i == 1) + (j == 1);
      const T P = p[j][i] * p[j][i] + (mid == 0 ? eta4 : mid == 1 ? eta16 : eta64), Q = q[j][i] * q[j][i];
      z[0][j] = P + T(1. / 3.) * Q;
      z[1][j] = p[j][i] * q[j][i];
      z[2][j] = P + T(.6) * Q;
    }
#pragma unroll
    for (int r = 0; r < 3; r++) {
      const T S = z[r][0] + z[r][2];
      zx[r][0][i] = S + z[r][1];
      zx[r][1][i] = z[r][2] - z[r][0];
      zx[r][2][i] = S + T(1. / 3.) * z[r][1];  // times 0.6
    }
  }
#pragma unroll
  for (int r = 0; r < 3; r++) {
    const double cz = r == 0 ? 1. : r == 1 ? 2. / 3. : 1. / 3.;
#pragma unroll
    for (int b = 0; b < 3; b++) {
      const double cy = b == 2 ? .6 : 1.;
      const T *f = zx[r][b];
      const T S = f[0] + f[2];
      M[0][b][r] = (Ek * T(cz * cy)) * (S + f[1]);
      if (!(b == 2 && r == 2)) M[1][b][r] = (Ek * T(cz * cy)) * (f[2] - f[0]);
      if (!(b == 2 && r > 0) && !(r == 2 && b > 0)) M[2][b][r] = (Ek * T(cz * cy * .6)) * (S + T(1. / 3.) * f[1]);
    }
  }
}

// what the element needs of one layer: 7 modal sums per component (index 0,
// the mean, does not enter)
template <typename T>
__device__ __forceinline__ void um_modes(const UFace<T> &B, const UFace<T> &F, T (&U)[3][8]) {
#pragma unroll
  for (int c = 0; c < 3; c++) {
    U[c][0] = T(0);
    U[c][1] = F.x[c] + B.x[c];
    U[c][5] = F.x[c] - B.x[c];
    U[c][2] = F.y[c] + B.y[c];
    U[c][6] = F.y[c] - B.y[c];
    U[c][3] = F.w[c] + B.w[c];
    U[c][7] = F.w[c] - B.w[c];
    U[c][4] = T(4) * (F.a[c] - B.a[c]) + (F.s[c] - B.s[c]);
  }
}

// R[i] of component c: the modal dual of the element's nodal forces (the force
// at a corner is the signed sum of the R[i]).  With D_cd the derivative d of
// component c (its four modes holding variable d):
//   test d of component d:  M_dd k2_d D_dd + sum_{e != d} M_de kl_de D_ee
//   test d of component c:  M_dd kx_dd D_cd + M_dc kx_dc D_dc
// CUBIC: kx = 1, one kl, one k2.
template <bool CUBIC, typename T>
__device__ __forceinline__ void um_force(const T (&M)[3][3][3], const T (&U)[3][8], const UModal<T> &m, int c,
                                         T (&R)[8]) {
#pragma unroll
  for (int i = 0; i < 8; i++) R[i] = T(0);
#pragma unroll
  for (int d = 0; d < 3; d++)
#pragma unroll
    for (int e = 0; e < 3; e++) {
      // trial derivative e: of component c (e == d), else of component e
      // (c == d) or, for c != d, only e == c of component d
      if (d != c && e != d && e != c) continue;
      const int cu = e == d ? c : c == d ? e : d;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        if (!um_pow(j, e)) continue;
        const T t = CUBIC && c != d ? U[cu][j]
                    : CUBIC         ? (e == d ? m.k2[0] : m.kl[0][0]) * U[cu][j]
                                    : (c != d ? m.kx[d][e] : e == d ? m.k2[d] : m.kl[d][e]) * U[cu][j];
#pragma unroll
        for (int i = 0; i < 8; i++)
          if (um_pow(i, d))
            R[i] += M[um_exp(i, d, j, e, 0)][um_exp(i, d, j, e, 1)][um_exp(i, d, j, e, 2)] * t;
      }
    }
}
// The same for s = 1 (the coarse multigrid levels): the odd moments vanish and
// the even ones are constants, so each block is diagonal (60 FMAs); Ek = E kap
// with the unit form's kap.
template <bool CUBIC, typename T>
__device__ __forceinline__ void um_force_unit(T Ek, const T (&U)[3][8], const UModal<T> &m, int c, T (&R)[8]) {
#pragma unroll
  for (int i = 0; i < 8; i++) R[i] = T(0);
#pragma unroll
  for (int d = 0; d < 3; d++)
#pragma unroll
    for (int e = 0; e < 3; e++) {
      if (d != c && e != d && e != c) continue;
      const int cu = e == d ? c : c == d ? e : d;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        if (!um_pow(j, e)) continue;
#pragma unroll
        for (int i = 0; i < 8; i++) {
          if (!um_pow(i, d)) continue;
          const int q0 = um_exp(i, d, j, e, 0), q1 = um_exp(i, d, j, e, 1), q2 = um_exp(i, d, j, e, 2);
          if ((q0 & 1) || (q1 & 1) || (q2 & 1)) continue;
          const T w = T((q0 ? 1. / 3. : 1.) * (q1 ? 1. / 3. : 1.) * (q2 ? 1. / 3. : 1.));
          const T k = CUBIC ? (c != d ? T(1) : e == d ? m.k2[0] : m.kl[0][0])
                            : (c != d ? m.kx[d][e] : e == d ? m.k2[d] : m.kl[d][e]);
          R[i] += (w * k) * U[cu][j];
        }
      }
    }
#pragma unroll
  for (int i = 1; i < 8; i++) R[i] *= Ek;
}

// One layer of an element column: the modal forces of the bottom face added to
// tot, those of the top face set in carry (per component s, x, y, w).
// UNIT: s = 1 (vb, vt unused).  CUBIC: elements whose three spacings agree
// (UModal::cubic): products by 1 and shared ones are left out, 590 FP64
// instructions per element and layer against 686; results are bitwise those of
// the general form.  A branch inside the element would keep
// all of it live at once (FP64: 23 registers spilled), so the kernels come in
// both forms (FP64 94 -> 86 us at 128^3, 620 -> 560 us at 256^3; FP32
// smoothing 72 -> 66 us at 128^3).
// Bound by instruction issue: with about 90 other vector instructions (counted in
// the assembly) the cubic form takes 0.64 of the issue slots at 128^3 and 0.67 at
// 256^3 (SQ counters; two waves per SIMD in FP64, three to four in FP32).  Against the 27-point form on the same tiles,
// general elements: FP64 176 -> 94 us at 128^3 and 1299 -> 640 us at 256^3, FP32
// 98 -> 59 us and 776 -> 391 us.
template <typename T, bool UNIT, bool CUBIC = false>
__device__ __forceinline__ void um_layer(const UFace<T> &B, const UFace<T> &F, const T *vb, const T *vt, T Ee,
                                         const UModal<T> &m, T (&tot)[3][4], T (&carry)[3][4]) {
  T U[3][8], M[3][3][3];
  const T Ek = Ee * m.kap;
  if constexpr (!UNIT) um_moments<T>(vb, vt, Ek, m.eta4, M);
  um_modes<T>(B, F, U);
#pragma unroll
  for (int c = 0; c < 3; c++) {
    T R[8];
    if constexpr (UNIT) um_force_unit<CUBIC>(Ek, U, m, c, R);
    else um_force<CUBIC>(M, U, m, c, R);
    tot[c][0] -= R[4];
    tot[c][1] += R[1] - R[5];
    tot[c][2] += R[2] - R[6];
    tot[c][3] += R[3] - R[7];
    carry[c][0] = R[4];
    carry[c][1] = R[1] + R[5];
    carry[c][2] = R[2] + R[6];
    carry[c][3] = R[3] + R[7];
  }
}

}  // namespace vfg
