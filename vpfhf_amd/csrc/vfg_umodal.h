// vfg_umodal.h -- the damaged-elasticity element in moment form, and the
// z-march that applies it.
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
// points with nine stress entries each: about 680 operations per element
// against 1390.  The moments themselves are Simpson sums of s over the
// 3 x 3 x 3 points {-1, 0, 1} (z in closed form), where v needs additions only.
//
// Scaling: a pair of derivatives d, e carries hx^2 / (h_d h_e) (and its Lame
// ratio) as one constant, rounded once; kap = vol mu / (16 hx^2) times the
// constants of the moment sums.
#pragma once
#include "vfg_internal.h"

namespace vfg {

// launch constants of the element in moment form
template <typename T>
struct UModal {
  T kap;         // vol mu1 / (2304 hx^2): 1/16 (derivatives) x 1/4 (v sums) x 1/36 (Simpson in x and y); unit: / 16
  T eta4;        // 4 eta
  // hx^2 / (h_d h_e) times 1 (kx), lam / mu (kl), and for d = e lam / mu + 2 (k2)
  T kx[3][3], kl[3][3], k2[3];
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

// exponents: modal index i = a + 2 b + 4 c of xi^a eta^b zeta^c
constexpr int um_pow(int i, int d) { return (i >> d) & 1; }
// exponent of variable e in (modal i without d) * (modal j without dp)
constexpr int um_exp(int i, int d, int j, int dp, int e) {
  return (e == d ? 0 : um_pow(i, e)) + (e == dp ? 0 : um_pow(j, e));
}

// the moments of s = v^2 + eta times E, M[p][q][r], from v at the corners of the
// bottom (vb) and top (vt) faces; Ek = E kap.  A point between two corners
// holds their sum (v twice, s four times), the face centre the sum of four, so
// Simpson's middle weight 4 is already in the value.
template <typename T>
__device__ __forceinline__ void um_moments(const T (&vb)[4], const T (&vt)[4], T Ek, T eta4, T (&M)[3][3][3]) {
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
template <typename T>
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
        const T t = (c != d ? m.kx[d][e] : e == d ? m.k2[d] : m.kl[d][e]) * U[cu][j];
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
template <typename T>
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
          R[i] += (w * (c != d ? m.kx[d][e] : e == d ? m.k2[d] : m.kl[d][e])) * U[cu][j];
        }
      }
    }
#pragma unroll
  for (int i = 1; i < 8; i++) R[i] *= Ek;
}

// ops whose store reads data of the owned node define own_load(n)
template <class Op, class = void>
struct ownm_of {
  using type = int;
};
template <class Op>
struct ownm_of<Op, std::void_t<decltype(&Op::own_load)>> {
  using type = decltype(std::declval<const Op &>().own_load(int64_t(0)));
};

// the value of the next lane of a 16-lane row (0 in the last one)
__device__ __forceinline__ float lane_up(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x101, 0xf, 0xf, true));  // row_shl:1
}
__device__ __forceinline__ double lane_up(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x101, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x101, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// faces (bits 0-5: X0..Z1) a node lies on
__device__ __forceinline__ uint32_t face_bits_xy(const Grid &G, int i, int j) {
  return (i == 0 ? 1u : 0u) | (i == G.nx - 1 ? 2u : 0u) | (j == 0 ? 4u : 0u) | (j == G.ny - 1 ? 8u : 0u);
}
// on_dirichlet from the face bits
__device__ __forceinline__ bool face_dirichlet(uint8_t face, uint8_t vert, uint32_t fb) {
  bool m = (face & fb) != 0u;
  if (vert && (fb & 3u) && (fb & 12u) && (fb & 48u))
    m = m || ((vert >> ((fb >> 1 & 1u) + 2u * (fb >> 3 & 1u) + 4u * (fb >> 5 & 1u))) & 1);
  return m;
}

// The z-march of the element in moment form: tiles, ownership and node order
// of march() (a 256- or 64-thread workgroup owns TX-1 x TY-1 node columns and
// recomputes a one-element halo), but
//   - a thread keeps the two node planes of its element as face sums (19
//     values), not corners, and the node plane under construction as modal
//     sums: an element adds its bottom part to the carried plane, and only
//     that one plane is turned into nodal values and combined with the x and y
//     neighbours per layer (lane shift along x, LDS along y);
//   - the y-combination and the store of a plane happen after the next
//     layer's barrier, so a layer has one barrier (s_in and s_red alternate
//     between two buffers: a buffer is written again two barriers after its
//     last read).
// Bound by instruction issue: about 690 FP64 and 140 other vector instructions
// per element and layer, 0.75 of the issue peak at 256^3 (two waves per SIMD in
// FP64, three to four in FP32).  Against the 27-point form on the same tiles:
// FP64 176 -> 94 us at 128^3 and 1299 -> 666 us at 256^3, FP32 98 -> 59 us and
// 776 -> 391 us.
// Op interface:
//   static constexpr bool UNIT        s = 1, no nodal v (coarse levels)
//   T load(f, n)                      f < 3: displacement; 3: v
//   T young(ex, ey, ek)               E_e, read one layer ahead
//   UModal<T> m; Grid G
//   O own_load(n)                     (has_own) data of an owned node, read a layer before its store
//   store(n, fb, acc, own[, o])       fb: face bits of the node; own: its displacement
//   partial(slot, sum)                (has_red) as in march()
template <typename T, int TX, int TY, class Op>
__device__ __forceinline__ void march_modal(const Grid &G, const Op &op, int OZ, int bx, int by, int bz,
                                            int rslot = 0) {
  static_assert(TX == 8 || TX == 16, "the x-combination shifts inside 16-lane rows");
  constexpr int NF = Op::UNIT ? 3 : 4;
  constexpr int NT = TX * TY, OX = TX - 1, OY = TY - 1, SX = TX + 1, PL = SX * (TY + 1);
  constexpr int NPF = (PL + NT - 1) / NT;
  constexpr bool RED = has_red<Op>::value, OWN = has_own<Op>::value;
  __shared__ T s_in[2][NF][PL];
  __shared__ T s_red[2][3][NT];
  const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
  const int ox0 = bx * OX, oy0 = by * OY, oz0 = bz * OZ;
  const int ex = ox0 - 1 + tx, ey = oy0 - 1 + ty;
  const bool exy_ok = ex >= 0 && ex < G.nex && ey >= 0 && ey < G.ney;
  const bool owner = tx < OX && ty < OY && (ox0 + tx) < G.nx && (oy0 + ty) < G.ny;
  const int64_t plane = (int64_t)G.nx * G.ny;
  const int64_t nxy = (int64_t)(ox0 + tx) + (int64_t)G.nx * (oy0 + ty);
  const uint32_t fbxy = face_bits_xy(G, ox0 + tx, oy0 + ty);

  int64_t soff[NPF];
  bool sok[NPF];
#pragma unroll
  for (int q = 0; q < NPF; q++) {
    const int n = tid + q * NT;
    const int gx = ox0 - 1 + n % SX, gy = oy0 - 1 + n / SX;
    sok[q] = n < PL && gx >= 0 && gx < G.nx && gy >= 0 && gy < G.ny;
    soff[q] = sok[q] ? (int64_t)gx + (int64_t)G.nx * gy : 0;
  }
  T pf[NPF][NF];
  auto fetch = [&](int iz) {
    const bool zok = iz >= 0 && iz < G.nz;  // uniform
#pragma unroll
    for (int q = 0; q < NPF; q++) {
      const bool ok = zok && sok[q];
      const int64_t nd = soff[q] + plane * iz;
#pragma unroll
      for (int f = 0; f < NF; f++) pf[q][f] = ok ? op.load(f, nd) : T(0);
    }
  };
  auto commit = [&](int b) {
#pragma unroll
    for (int q = 0; q < NPF; q++) {
      const int n = tid + q * NT;
      if (n < PL)
#pragma unroll
        for (int f = 0; f < NF; f++) s_in[b][f][n] = pf[q][f];
    }
  };
  struct Plane {
    UFace<T> f;
    T v[4], own[3];
  };
  const int c0 = ty * SX + tx;
  auto read_plane = [&](int b, Plane &P) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const T x0 = s_in[b][c][c0], x1 = s_in[b][c][c0 + 1], x2 = s_in[b][c][c0 + SX], x3 = s_in[b][c][c0 + SX + 1];
      uface_set<T>(P.f, c, x0, x1, x2, x3);
      P.own[c] = x3;
    }
    if constexpr (!Op::UNIT)
#pragma unroll
      for (int q = 0; q < 4; q++) P.v[q] = s_in[b][NF - 1][c0 + (q >> 1) * SX + (q & 1)];
  };
  auto young = [&](int ek) -> T { return exy_ok && ek >= 0 && ek < G.nez ? op.young(ex, ey, ek) : T(0); };
  using OwnT = typename ownm_of<Op>::type;
  auto own_at = [&](int k) -> OwnT {
    OwnT o{};
    if constexpr (OWN)
      if (owner && k >= oz0 && k >= 0 && k < G.nz) o = op.own_load(nxy + plane * k);
    return o;
  };

  T carry[3][4];  // modal sums of the node plane on top of the last layer
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int q = 0; q < 4; q++) carry[c][q] = T(0);
  T pend[3], pown[3];  // this thread's part of the plane waiting for its y-combination, and its displacement
  OwnT po{};
  double racc = 0.;
  auto finish = [&](int k, int b) {
    if (!owner || k < oz0 || k < 0) return;
    T acc[3];
#pragma unroll
    for (int c = 0; c < 3; c++) acc[c] = pend[c] + s_red[b][c][tid + TX];
    const uint32_t fb = fbxy | (k == 0 ? 16u : 0u) | (k == G.nz - 1 ? 32u : 0u);
    const int64_t n = nxy + plane * k;
    if constexpr (OWN) {
      if constexpr (RED) racc += op.store(n, fb, acc, pown, po);
      else op.store(n, fb, acc, pown, po);
    } else {
      if constexpr (RED) racc += op.store(n, fb, acc, pown);
      else op.store(n, fb, acc, pown);
    }
  };
  const int ek0 = oz0 - 1, ek_end = min(oz0 + OZ - 1, G.nz - 1);
  // one element layer between node planes ek (B) and ek + 1 (Tp)
  auto layer = [&](int ek, const Plane &B, Plane &Tp, T &E_next) {
    const T Ee = E_next;
    const int b = (ek - ek0) & 1;
    commit(b ^ 1);  // plane ek + 1
    if (ek < ek_end) fetch(ek + 2);
    E_next = young(ek + 1);
    const OwnT on = own_at(ek);
    __syncthreads();
    read_plane(b ^ 1, Tp);
    if (ek > ek0) finish(ek - 1, b ^ 1);
    T tot[3][4];
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        tot[c][q] = carry[c][q];
        carry[c][q] = T(0);
      }
    if (exy_ok && ek >= 0 && ek < G.nez) {
      T U[3][8], M[3][3][3];
      const T Ek = Ee * op.m.kap;
      if constexpr (!Op::UNIT) um_moments<T>(B.v, Tp.v, Ek, op.m.eta4, M);
      um_modes<T>(B.f, Tp.f, U);
#pragma unroll
      for (int c = 0; c < 3; c++) {
        T R[8];
        if constexpr (Op::UNIT) um_force_unit<T>(Ek, U, op.m, c, R);
        else um_force<T>(M, U, op.m, c, R);
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
    // node (ex + 1, ey + 1): corner x1 of this element and x0 of the next lane's
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const T s0 = (tot[c][0] + tot[c][1]) + lane_up(tot[c][0] - tot[c][1]);
      const T s1 = (tot[c][2] + tot[c][3]) + lane_up(tot[c][2] - tot[c][3]);
      pend[c] = s0 + s1;             // corner y1
      s_red[b][c][tid] = s0 - s1;    // corner y0, for the element row below
      pown[c] = B.own[c];
    }
    po = on;
  };

  Plane pa, pb;
  fetch(ek0);
  commit(0);
  fetch(ek0 + 1);
  T E_next = young(ek0);
  __syncthreads();
  read_plane(0, pa);
  int ek = ek0;
  for (; ek <= ek_end; ek += 2) {
    layer(ek, pa, pb, E_next);
    if (ek + 1 > ek_end) break;
    layer(ek + 1, pb, pa, E_next);
  }
  __syncthreads();
  finish(ek_end, (ek_end - ek0) & 1);
  if constexpr (RED) {
    __shared__ double s_rs[NT / 64];
    const double v = block_sum<NT>(racc, s_rs);
    if (tid == 0) op.partial(rslot, v);
  }
}
template <typename T, int TX, int TY, class Op>
__device__ __forceinline__ void march_modal(const Grid &G, const Op &op, int OZ, Blk3 b, int rslot = 0) {
  march_modal<T, TX, TY>(G, op, OZ, b.x, b.y, b.z, rslot);
}

}  // namespace vfg
