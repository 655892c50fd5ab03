// vfg_u.hip -- u-subproblem operators on gfx950.
//
// Element bilinear form (VF_BilinearFormU3D_local, VFMech.c:227-290):
//   Ke[(a,c1),(b,c2)] = sum_g W_g s_g [lam d_c1 phi_a d_c2 phi_b
//                                      + mu d_c2 phi_a d_c1 phi_b
//                                      + delta_c1c2 mu grad phi_a . grad phi_b]
//   s_g = v_g^2 + eta.
// Applied matrix-free: (Ke x)_{a,c} = sum_g sum_d sigma_cd(g) d_d phi_a(g) with
//   sigma = W s (lam tr(H) I + mu (H + H^T)),  H_cd = d_d u_c  (displacement
//   gradient of x).  Without compression the sum over the 27 points is taken
// in closed form from polynomial moments of s and the modal sums of x
// (vfg_umodal.h); the compressed and the stored-coefficient forms visit the
// points by sum factorisation with the 1-D Gauss tables.
#include "vfg_internal.h"
#include "vfg_umodal.h"
#include "vfg_kernels.h"
#include "vfg_batch_apply.h"
#include "vfg_handle.h"
#include "vfg_mg.h"
#include "vfg_bmg.h"

namespace vfg {

// Apply of one element under UNILATERAL_NOCOMPRESSION (VFMech.c:299-376): X
// holds (x0,x1,x2,v) at the 8 corners, cE = E_e * hx*hy*hz, lam1/mu1 are the
// Lame constants for E = 1.  The gradients are carried pre-scaled by mu
// (H' = mu H), so that
//   sigma / (W s cE) = lr tr(H') I + H' + H'^T,  lr = lam / mu,
// and each stress entry is accumulated with one FMA by its weight W s cE; at
// the Gauss points set in cm the spherical part keeps kappa (1 + eta) instead
// of kappa s, i.e.
//   sigma / (W cE) = (kr - 2 s / 3) tr(H') I + s (H' + H'^T),
//   kr = kappa (1 + eta) / mu = (lr + 2/3)(1 + eta).
template <typename T>
__device__ __forceinline__ void u_elem_apply(const T (&X)[2][4][4], T cE, T lam1, T mu1, T eta,
                                             T ihx, T ihy, T ihz, T (&r)[8][3], uint32_t cm) {
  const T lr = lam1 / mu1;
  const T kr = (lr + T(2. / 3.)) * (T(1) + eta);
  const T mx = mu1 * ihx, my = mu1 * ihy, mz = mu1 * ihz;
  // differences along each direction, scaled by mu/h
  T Dx[3][2][2], Dy[3][2][2], Dz[3][2][2];  // Dx[c][k][j], Dy[c][k][i], Dz[c][j][i]
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
      for (int q = 0; q < 2; q++) {
        Dx[c][p][q] = (X[p][q * 2 + 1][c] - X[p][q * 2 + 0][c]) * mx;
        Dy[c][p][q] = (X[p][2 + q][c] - X[p][q][c]) * my;
        Dz[c][p][q] = (X[1][p * 2 + q][c] - X[0][p * 2 + q][c]) * mz;
      }
  // mu d_z u_c at (gx,gy): constant in z
  T Gz[3][3][3];  // [c][gy][gx]
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int gx = 0; gx < 3; gx++) {
      T a0 = interp<T>(gx, Dz[c][0][0], Dz[c][0][1]);
      T a1 = interp<T>(gx, Dz[c][1][0], Dz[c][1][1]);
#pragma unroll
      for (int gy = 0; gy < 3; gy++) Gz[c][gy][gx] = interp<T>(gy, a0, a1);
    }
  // v interpolated in x and y on both z-faces
  T vxy[2][3][3];  // [k][gy][gx]
#pragma unroll
  for (int k = 0; k < 2; k++)
#pragma unroll
    for (int gx = 0; gx < 3; gx++) {
      T a0 = interp<T>(gx, X[k][0][3], X[k][1][3]);
      T a1 = interp<T>(gx, X[k][2][3], X[k][3][3]);
#pragma unroll
      for (int gy = 0; gy < 3; gy++) vxy[k][gy][gx] = interp<T>(gy, a0, a1);
    }

  T Rx[3][2][2], Ry[3][2][2], Sz[3][3][3];  // Rx[c][k][j], Ry[c][k][i], Sz[c][gy][gx]
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
      for (int q = 0; q < 2; q++) Rx[c][p][q] = Ry[c][p][q] = T(0);
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int gy = 0; gy < 3; gy++)
#pragma unroll
      for (int gx = 0; gx < 3; gx++) Sz[c][gy][gx] = T(0);

#pragma unroll
  for (int gz = 0; gz < 3; gz++) {
    T Gx[3][3], Gy[3][3];  // Gx[c][gy], Gy[c][gx]
#pragma unroll
    for (int c = 0; c < 3; c++) {
      T bx0 = interp<T>(gz, Dx[c][0][0], Dx[c][1][0]);
      T bx1 = interp<T>(gz, Dx[c][0][1], Dx[c][1][1]);
      T by0 = interp<T>(gz, Dy[c][0][0], Dy[c][1][0]);
      T by1 = interp<T>(gz, Dy[c][0][1], Dy[c][1][1]);
#pragma unroll
      for (int g = 0; g < 3; g++) {
        Gx[c][g] = interp<T>(g, bx0, bx1);
        Gy[c][g] = interp<T>(g, by0, by1);
      }
    }
    T Sx[3][3], Sy[3][3];  // Sx[c][gy] = sum_gx sigma_c0, Sy[c][gx] = sum_gy sigma_c1
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int g = 0; g < 3; g++) Sx[c][g] = Sy[c][g] = T(0);
    const T wz = cE * T(gW(gz));
#pragma unroll
    for (int gy = 0; gy < 3; gy++) {
      const T wzy = wz * T(gW(gy));
#pragma unroll
      for (int gx = 0; gx < 3; gx++) {
        const T v = interp<T>(gz, vxy[0][gy][gx], vxy[1][gy][gx]);
        const T wq = wzy * T(gW(gx));
        const T cq = wq * (v * v + eta);
        const T H00 = Gx[0][gy], H01 = Gy[0][gx], H02 = Gz[0][gy][gx];
        const T H10 = Gx[1][gy], H11 = Gy[1][gx], H12 = Gz[1][gy][gx];
        const T H20 = Gx[2][gy], H21 = Gy[2][gx], H22 = Gz[2][gy][gx];
        const T t01 = H01 + H10, t02 = H02 + H20, t12 = H12 + H21;
        const bool comp = (cm >> ((gz * 3 + gy) * 3 + gx)) & 1u;
        const T lw = comp ? wq * (kr - T(2. / 3.) * (v * v + eta)) : cq * lr;
        const T L = lw * (H00 + H11 + H22);
        const T c2 = cq + cq;
        Sx[0][gy] += L + c2 * H00; Sx[1][gy] += cq * t01; Sx[2][gy] += cq * t02;
        Sy[0][gx] += cq * t01; Sy[1][gx] += L + c2 * H11; Sy[2][gx] += cq * t12;
        Sz[0][gy][gx] += cq * t02; Sz[1][gy][gx] += cq * t12; Sz[2][gy][gx] += L + c2 * H22;
      }
    }
    const T pz0 = T(gP0(gz)), pz1 = T(gP1(gz));
#pragma unroll
    for (int c = 0; c < 3; c++) {
      T ax0 = T(0), ax1 = T(0), ay0 = T(0), ay1 = T(0);
#pragma unroll
      for (int g = 0; g < 3; g++) {
        ax0 += T(gP0(g)) * Sx[c][g]; ax1 += T(gP1(g)) * Sx[c][g];
        ay0 += T(gP0(g)) * Sy[c][g]; ay1 += T(gP1(g)) * Sy[c][g];
      }
      Rx[c][0][0] += pz0 * ax0; Rx[c][0][1] += pz0 * ax1;
      Rx[c][1][0] += pz1 * ax0; Rx[c][1][1] += pz1 * ax1;
      Ry[c][0][0] += pz0 * ay0; Ry[c][0][1] += pz0 * ay1;
      Ry[c][1][0] += pz1 * ay0; Ry[c][1][1] += pz1 * ay1;
    }
  }
  // project Sz onto the bilinear basis in (x,y); scale each direction by 1/h once
#pragma unroll
  for (int c = 0; c < 3; c++) {
    T b[3][2];  // [gy][i]
#pragma unroll
    for (int gy = 0; gy < 3; gy++) {
      T a0 = T(0), a1 = T(0);
#pragma unroll
      for (int gx = 0; gx < 3; gx++) { a0 += T(gP0(gx)) * Sz[c][gy][gx]; a1 += T(gP1(gx)) * Sz[c][gy][gx]; }
      b[gy][0] = a0; b[gy][1] = a1;
    }
    T Rz[2][2];  // [j][i]
#pragma unroll
    for (int i = 0; i < 2; i++) {
      T a0 = T(0), a1 = T(0);
#pragma unroll
      for (int gy = 0; gy < 3; gy++) { a0 += T(gP0(gy)) * b[gy][i]; a1 += T(gP1(gy)) * b[gy][i]; }
      Rz[0][i] = a0 * ihz; Rz[1][i] = a1 * ihz;
    }
    T sx[2][2], sy[2][2];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
      for (int q = 0; q < 2; q++) { sx[p][q] = Rx[c][p][q] * ihx; sy[p][q] = Ry[c][p][q] * ihy; }
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
          const T vx = i ? sx[k][j] : -sx[k][j];
          const T vy = j ? sy[k][i] : -sy[k][i];
          const T vz = k ? Rz[j][i] : -Rz[j][i];
          r[(k * 2 + j) * 2 + i][c] = vx + vy + vz;
        }
  }
}

// The same element apply for march_lds: the corners are re-read from LDS in
// every Gauss layer gz (xs(k, q, f)), so that only one layer's
// interpolants are live and the FP64 kernel fits 256 registers (two waves
// per SIMD).  Per layer: the corners interpolated to the layer (Uz, Vz) and
// their z-differences (Dz); x-derivatives Gx[c][gy] for the layer; then
// gx-outer, gy-inner over the 9 points, with interpolation written as
// a + p1 (b - a) (one FMA per point and value).  Accumulation and the final
// projections are those of u_elem_apply.  Stored coefficients: the 27 products
// W_g s_g E_e vol of the element are read from QS[g * QSTRIDE],
// g = (gz * 3 + gy) * 3 + gx.
template <int QSTRIDE, typename T, typename XS, typename OUT>
__device__ __forceinline__ void u_elem_apply_lds_stored(const XS &xs, T lam1, T mu1, T ihx, T ihy, T ihz,
                                                        const OUT &out, const T *__restrict__ QS) {
  const T lr = lam1 / mu1;
  const T mx = mu1 * ihx, my = mu1 * ihy, mz = mu1 * ihz;
  // Rx[c][k][j], Ry[c][k][i]; Sz[c][gy][i]: the z-stress summed over the Gauss
  // layers and projected onto x at once (18 accumulators rather than 27: the
  // element then fits two waves per SIMD without spilling)
  T Rx[3][2][2], Ry[3][2][2], Sz[3][3][2];
#pragma unroll
  for (int c = 0; c < 3; c++) {
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
      for (int q = 0; q < 2; q++) Rx[c][p][q] = Ry[c][p][q] = T(0);
#pragma unroll
    for (int p = 0; p < 3; p++)
#pragma unroll
      for (int q = 0; q < 2; q++) Sz[c][p][q] = T(0);
  }
#pragma unroll
  for (int gz = 0; gz < 3; gz++) {
    const T pz0 = T(gP0(gz)), pz1 = T(gP1(gz));
    // compiler barrier: the corners are read again from LDS for this layer
    // rather than kept live across layers
    asm volatile("" ::: "memory");
    T Dz[4][3], Gx[3][3], by0[3], byd[3];
    T Ql[3][3];  // stored coefficients of the layer [gx][gy]
#pragma unroll
    for (int gx = 0; gx < 3; gx++)
#pragma unroll
      for (int gy = 0; gy < 3; gy++) Ql[gx][gy] = QS[((gz * 3 + gy) * 3 + gx) * QSTRIDE];
    {
      T Uz[4][3];
#pragma unroll
      for (int q = 0; q < 4; q++) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
          const T a = xs(0, q, c), d = xs(1, q, c) - a;
          Uz[q][c] = a + pz1 * d;
          Dz[q][c] = d * mz;
        }
      }
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const T bx0 = (Uz[1][c] - Uz[0][c]) * mx, bxd = (Uz[3][c] - Uz[2][c]) * mx - bx0;
#pragma unroll
        for (int gy = 0; gy < 3; gy++) Gx[c][gy] = bx0 + T(gP1(gy)) * bxd;
        by0[c] = (Uz[2][c] - Uz[0][c]) * my;
        byd[c] = (Uz[3][c] - Uz[1][c]) * my - by0[c];
      }
    }
    T Dzx0[3], Dzx2[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
      Dzx0[c] = Dz[1][c] - Dz[0][c];
      Dzx2[c] = Dz[3][c] - Dz[2][c];
    }
    T Sx[3][3], ay[3][2];  // Sx[c][gy] = sum_gx sigma_c0; ay[c][i] = y-projection of sum_gy sigma_c1
#pragma unroll
    for (int c = 0; c < 3; c++) {
#pragma unroll
      for (int g = 0; g < 3; g++) Sx[c][g] = T(0);
      ay[c][0] = ay[c][1] = T(0);
    }
#pragma unroll
    for (int gx = 0; gx < 3; gx++) {
      const T px = T(gP1(gx));
      T Gy[3], az0[3], azd[3], Sy[3];
#pragma unroll
      for (int c = 0; c < 3; c++) {
        Gy[c] = by0[c] + px * byd[c];
        az0[c] = Dz[0][c] + px * Dzx0[c];
        azd[c] = Dz[2][c] + px * Dzx2[c] - az0[c];
        Sy[c] = T(0);
      }
#pragma unroll
      for (int gy = 0; gy < 3; gy++) {
        const T cq = Ql[gx][gy];
        const T H00 = Gx[0][gy], H01 = Gy[0], H02 = az0[0] + T(gP1(gy)) * azd[0];
        const T H10 = Gx[1][gy], H11 = Gy[1], H12 = az0[1] + T(gP1(gy)) * azd[1];
        const T H20 = Gx[2][gy], H21 = Gy[2], H22 = az0[2] + T(gP1(gy)) * azd[2];
        const T t01 = H01 + H10, t02 = H02 + H20, t12 = H12 + H21;
        const T lt = lr * (H00 + H11 + H22);
        const T t00 = lt + T(2) * H00, t11 = lt + T(2) * H11, t22 = lt + T(2) * H22;
        Sx[0][gy] += cq * t00; Sx[1][gy] += cq * t01; Sx[2][gy] += cq * t02;
        Sy[0] += cq * t01; Sy[1] += cq * t11; Sy[2] += cq * t12;
        const T z0 = cq * t02, z1 = cq * t12, z2 = cq * t22;
        Sz[0][gy][0] += T(gP0(gx)) * z0; Sz[0][gy][1] += T(gP1(gx)) * z0;
        Sz[1][gy][0] += T(gP0(gx)) * z1; Sz[1][gy][1] += T(gP1(gx)) * z1;
        Sz[2][gy][0] += T(gP0(gx)) * z2; Sz[2][gy][1] += T(gP1(gx)) * z2;
      }
#pragma unroll
      for (int c = 0; c < 3; c++) {
        ay[c][0] += T(gP0(gx)) * Sy[c];
        ay[c][1] += T(gP1(gx)) * Sy[c];
      }
    }
#pragma unroll
    for (int c = 0; c < 3; c++) {
      T ax0 = T(0), ax1 = T(0);
#pragma unroll
      for (int g = 0; g < 3; g++) { ax0 += T(gP0(g)) * Sx[c][g]; ax1 += T(gP1(g)) * Sx[c][g]; }
      Rx[c][0][0] += pz0 * ax0; Rx[c][0][1] += pz0 * ax1;
      Rx[c][1][0] += pz1 * ax0; Rx[c][1][1] += pz1 * ax1;
      Ry[c][0][0] += pz0 * ay[c][0]; Ry[c][0][1] += pz0 * ay[c][1];
      Ry[c][1][0] += pz1 * ay[c][0]; Ry[c][1][1] += pz1 * ay[c][1];
    }
  }
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const T (&b)[3][2] = Sz[c];  // [gy][i]
    T Rz[2][2];  // [j][i]
#pragma unroll
    for (int i = 0; i < 2; i++) {
      T a0 = T(0), a1 = T(0);
#pragma unroll
      for (int gy = 0; gy < 3; gy++) { a0 += T(gP0(gy)) * b[gy][i]; a1 += T(gP1(gy)) * b[gy][i]; }
      Rz[0][i] = a0 * ihz; Rz[1][i] = a1 * ihz;
    }
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
          const T vx = (i ? Rx[c][k][j] : -Rx[c][k][j]) * ihx;
          const T vy = (j ? Ry[c][k][i] : -Ry[c][k][i]) * ihy;
          const T vz = k ? Rz[j][i] : -Rz[j][i];
          out((k * 2 + j) * 2 + i, c, vx + vy + vz);
        }
  }
}

// NOCOMPRESSION apply (Gauss-point form: its branch is per point)
template <typename T>
struct UAuxM {
  T E;
  uint32_t m;  // compressed Gauss points of the Jacobian state
};

template <typename T>
struct UApplyUniOp {
  static constexpr int NF = 4, NC = 3;
  const T *x;
  T *y;
  const T *v;
  const double *E_elem;
  const uint32_t *cmask;
  Grid G;
  BcMask bc;
  T E, lam1, mu1, eta, vol, ihx, ihy, ihz;
  __device__ T load(int f, int64_t n) const { return f < 3 ? x[3 * n + f] : v[n]; }
  __device__ UAuxM<T> aux(int ex, int ey, int ek) const {
    const int64_t c = cell_id(G, ex, ey, ek);
    return UAuxM<T>{E_elem ? T(E_elem[c]) : E, cmask[c]};
  }
  __device__ void element(int, int, int, const T (&xin)[2][4][4], UAuxM<T> a, T (&r)[8][3]) const {
    u_elem_apply<T>(xin, a.E * vol, lam1, mu1, eta, ihx, ihy, ihz, r, a.m);
  }
  __device__ void store(int i, int j, int k, const T (&acc)[3], const T (&own)[4]) const {
    int64_t n = node_id(G, i, j, k);
#pragma unroll
    for (int c = 0; c < 3; c++)
      y[3 * n + c] = on_dirichlet(G, bc.face[c], bc.vert[c], i, j, k) ? own[c] : acc[c];
  }
};
// FP32: at most 256 registers, two waves per SIMD
template <typename T, int TX, int TY>
__global__ __launch_bounds__(TX *TY, sizeof(T) == 4 ? 2 : 1) void k_u_apply_uni(UApplyUniOp<T> op, int OZ) {
  march<T, TX, TY>(op.G, op, OZ, xcd_block());
}

// Apply in moment form (UNILATERAL_NONE).  UNIT: s = 1, the coarse multigrid
// levels; the record is the same for both, the kernel chooses.
template <typename T>
struct UModRec {
  const T *x;
  T *y;
  const T *v;
  const double *E_elem;
  Grid G;
  BcMask bc;
  T E;
  UModal<T> m;
};
// the parts of the march's interface that every moment-form operator shares
// (Rec: UModRec<T> or a record derived from it)
template <typename T_, bool UNIT, class Rec, bool CUBIC>
struct UModBase : Rec {
  using T = T_;
  using Record = Rec;
  static constexpr int NF = UNIT ? 3 : 4, NC = 3;
  struct Face {
    UFace<T> f;
    T v[UNIT ? 1 : 4], own[3];
  };
  struct Own {
    T x[3];
  };
  using Aux = T;  // E_e
  using Raw = T;
  static __device__ T off() { return T(0); }
  __device__ T stage(int, T v) const { return v; }
  template <class RD>
  __device__ void face(const RD &rd, Face &F) const {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const T x3 = rd(c, 3);
      uface_set<T>(F.f, c, rd(c, 0), rd(c, 1), rd(c, 2), x3);
      F.own[c] = x3;
    }
    if constexpr (!UNIT)
#pragma unroll
      for (int q = 0; q < 4; q++) F.v[q] = rd(NF - 1, q);
  }
  __device__ Own own(const Face &F) const { return Own{{F.own[0], F.own[1], F.own[2]}}; }
  __device__ T aux(int ex, int ey, int ek, int, int) const {
    return this->E_elem ? T(this->E_elem[cell_id(this->G, ex, ey, ek)]) : this->E;
  }
  __device__ void element(T Ee, const Face &B, const Face &F, T (&tot)[3][4], T (&carry)[3][4]) const {
    um_layer<T, UNIT, CUBIC>(B.f, F.f, B.v, F.v, Ee, this->m, tot, carry);
  }
  // A x of a node: the displacement itself on the Dirichlet rows (a wavefront
  // without a boundary node skips the tests)
  __device__ void rows(uint32_t fb, const T (&acc)[3], const Own &own, T (&yv)[3]) const {
#pragma unroll
    for (int c = 0; c < 3; c++) yv[c] = acc[c];
    if (__builtin_amdgcn_ballot_w64(fb != 0u) != 0) {
      __asm__ __volatile__("");  // keeps the tests inside the branch
#pragma unroll
      for (int c = 0; c < 3; c++)
        if (face_dirichlet(this->bc.face[c], this->bc.vert[c], fb)) yv[c] = own.x[c];
    }
  }
};
template <typename T, bool UNIT, bool CUBIC = false>
struct UModOp : UModBase<T, UNIT, UModRec<T>, CUBIC> {
  using typename UModBase<T, UNIT, UModRec<T>, CUBIC>::Own;
  __device__ T load(int f, int64_t n) const { return f < 3 ? this->x[3 * n + f] : this->v[n]; }
  __device__ void store(int64_t n, uint32_t fb, const T (&acc)[3], const Own &own) const {
    T yv[3];
    this->rows(fb, acc, own, yv);
#pragma unroll
    for (int c = 0; c < 3; c++) this->y[3 * n + c] = yv[c];
  }
};
template <typename T>
static void umod_fill(UModRec<T> &r, const DevProblem &P, const T *x, T *y) {
  r.x = x;
  r.y = y;
  r.v = sizeof(T) == 4 ? (const T *)(const void *)P.V32 : (const T *)(const void *)P.V;
  r.E_elem = P.E_elem;
  r.G = P.G;
  r.bc = P.bcU;
  r.E = T(P.E);
  r.m = make_umodal<T>(P.G, P.lam1, P.mu1, P.eta, P.unit != 0);
}

// waves per SIMD asked of the compiler: FP64 two (256 registers), FP32 three
template <typename T>
constexpr int um_waves() { return sizeof(T) == 8 ? 2 : 3; }
template <typename T, int TX, int TY, bool UNIT, bool CUBIC>
__global__ __launch_bounds__(TX *TY, um_waves<T>()) void k_u_apply(UModOp<T, UNIT, CUBIC> op, int OZ) {
  march_modal<TX, TY>(op.G, op, OZ, xcd_block());
}

// FP32 multigrid apply fused with its Chebyshev(1)-Jacobi step (mg_cheb_entry
// with one step, vfg_solve.hip's V-cycle):
//   pre  (from x = 0): x = c2 D^-1 b staged on the fly; stores x and the
//        residual b - A x (0 on the Dirichlet rows) for the restriction;
//   post: xo = x + c2 D^-1 (b - A x), A x = x on Dirichlet rows, into a
//        buffer other than x (neighbouring tiles still stage x); b and D^-1
//        of the owned node are loaded a node plane ahead (own_load).  The
//        rz form also reduces r . xo (r: the FP64 residual the V-cycle
//        preconditions) over the owned rows, one partial per workgroup.
struct UMgRec : UModRec<float> {
  const float *b, *dinv;
  float *xo, *ro;
  float c2;
  const double *r64;  // rz form
  double *part;       // rz form
};
template <bool UNIT, bool CUBIC = false>
struct UMgPreOp : UModBase<float, UNIT, UMgRec, CUBIC> {
  using typename UModBase<float, UNIT, UMgRec, CUBIC>::Own;
  struct Raw {
    float b, di;
  };
  static __device__ Raw off() { return Raw{0.f, 0.f}; }
  __device__ Raw load(int f, int64_t n) const {
    if (f == 3) return Raw{this->v[n], 0.f};
    return Raw{this->b[3 * n + f], this->dinv[3 * n + f]};
  }
  __device__ float stage(int f, const Raw &r) const { return f == 3 ? r.b : this->c2 * r.di * r.b; }
  struct OwnB {
    float b[3];
  };
  __device__ OwnB own_load(int64_t n) const { return OwnB{{this->b[3 * n], this->b[3 * n + 1], this->b[3 * n + 2]}}; }
  __device__ void store(int64_t n, uint32_t fb, const float (&acc)[3], const Own &own, const OwnB &o) const {
    const Own rhs{{o.b[0], o.b[1], o.b[2]}};
    float yv[3];
    this->rows(fb, acc, rhs, yv);  // b itself on the Dirichlet rows
#pragma unroll
    for (int c = 0; c < 3; c++) {
      this->xo[3 * n + c] = own.x[c];
      this->ro[3 * n + c] = o.b[c] - yv[c];
    }
  }
};
struct MgOwn {
  float b[3], di[3];
};
struct MgOwnR {
  float b[3], di[3];
  double r[3];
};
template <bool UNIT, bool RZ, bool CUBIC = false>
struct UMgPostOp : UModBase<float, UNIT, UMgRec, CUBIC> {
  using typename UModBase<float, UNIT, UMgRec, CUBIC>::Own;
  __device__ float load(int f, int64_t n) const { return f < 3 ? this->x[3 * n + f] : this->v[n]; }
  __device__ auto own_load(int64_t n) const {
    std::conditional_t<RZ, MgOwnR, MgOwn> o;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      o.b[c] = this->b[3 * n + c];
      o.di[c] = this->dinv[3 * n + c];
      if constexpr (RZ) o.r[c] = this->r64[3 * n + c];
    }
    return o;
  }
  template <typename O>
  __device__ auto store(int64_t n, uint32_t fb, const float (&acc)[3], const Own &own, const O &o) const {
    double rz = 0.;
    float yv[3];
    this->rows(fb, acc, own, yv);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const float z = own.x[c] + this->c2 * o.di[c] * (o.b[c] - yv[c]);
      this->xo[3 * n + c] = z;
      if constexpr (RZ) rz += o.r[c] * (double)z;
    }
    if constexpr (RZ) return rz;
  }
};
template <bool CUBIC>
struct UMgPostRzOp : UMgPostOp<false, true, CUBIC> {
  __device__ void partial(int slot, double v) const { this->part[slot] = v; }
};
template <class Op, int TX, int TY>
__global__ __launch_bounds__(TX *TY, 3) void k_u_mg(Op op, int OZ) {
  march_modal<TX, TY>(op.G, op, OZ, xcd_block(), blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z));
}

// the FP64 apply also reducing p.q (p = the input, q = the output, every
// row) to one partial per workgroup: the CG's p.q without another pass
template <bool CUBIC>
struct UApplyDotOp : UModOp<double, false, CUBIC> {
  using typename UModOp<double, false, CUBIC>::Own;
  double *part;
  __device__ double store(int64_t n, uint32_t fb, const double (&acc)[3], const Own &own) const {
    double d = 0., yv[3];
    this->rows(fb, acc, own, yv);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      this->y[3 * n + c] = yv[c];
      d += own.x[c] * yv[c];
    }
    return d;
  }
  __device__ void partial(int slot, double v) const { part[slot] = v; }
};
template <int W, bool CUBIC>
__global__ __launch_bounds__(W *W, 2) void k_u_apply_dot(UApplyDotOp<CUBIC> op, int OZ) {
  march_modal<W, W>(op.G, op, OZ, xcd_block(),
                      blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z));
}

// ------------------------------------------------ stored-form FP64 apply
// The stored form (variant B): q_g = W_g (v_g^2 + eta) E_e vol for the 27
// Gauss points of every element, the integrand weights of
// VF_BilinearFormU3D_local (VFMech.c:240-252), computed once per coefficient
// state (k_u_qsetup_lds) so that the apply stages only x.
// The stored form on the node-owned march (march_lds): 16 x 16 element slots
// per tile, (15 bx - 1 + tx, 15 by - 1 + ty), halo elements stored in every
// tile that computes them: [tile][element layer][27][256], the layout of the
// V operator's weights.
template <bool DOT>
struct UApplyLdsqOp {
  static constexpr int NF = 3, NC = 3;
  const double *x;
  double *y, *part;
  const double *uq;
  Grid G;
  BcMask bc;
  double lam1, mu1, ihx, ihy, ihz;
  __device__ double load(int f, int64_t n) const { return x[3 * n + f]; }
  template <typename XS>
  __device__ void element_lds(int, int, int ek, const XS &xs, double (&r)[8][3]) const {
    const int tile = blockIdx.x + gridDim.x * blockIdx.y;
    const double *q = uq + ((int64_t)tile * G.nez + ek) * 27 * 256 + threadIdx.x;
    u_elem_apply_lds_stored<256, double>(xs, lam1, mu1, ihx, ihy, ihz, [&](int a, int c, double v) { r[a][c] = v; },
                                         q);
  }
  __device__ auto store(int i, int j, int k, const double (&acc)[3], const double (&own)[3]) const {
    const int64_t n = node_id(G, i, j, k);
    double d = 0.;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const double yv = on_dirichlet(G, bc.face[c], bc.vert[c], i, j, k) ? own[c] : acc[c];
      y[3 * n + c] = yv;
      d += own[c] * yv;
    }
    if constexpr (DOT) return d;
  }
};
struct UApplyLdsqDotOp : UApplyLdsqOp<true> {
  __device__ void partial(int slot, double v) const { part[slot] = v; }
};
__global__ __launch_bounds__(256, 2) void k_u_apply_ldsq(UApplyLdsqOp<false> op, int OZ) {
  march_lds<double, 16, 16>(op.G, op, OZ, blockIdx.x, blockIdx.y, blockIdx.z);
}
__global__ __launch_bounds__(256, 2) void k_u_apply_ldsq_dot(UApplyLdsqDotOp op, int OZ) {
  march_lds<double, 16, 16>(op.G, op, OZ, blockIdx.x, blockIdx.y, blockIdx.z,
                                   blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z));
}
// q of the node-owned tiles: block (bx, by, ek), thread = slot
__global__ __launch_bounds__(256) void k_u_qsetup_lds(Grid G, const double *__restrict__ V,
                                                      const double *__restrict__ E_elem, double E, double eta,
                                                      double *__restrict__ uq) {
  const int tid = threadIdx.x;
  const Blk3 b = xcd_block();
  const int ex = b.x * 15 - 1 + tid % 16, ey = b.y * 15 - 1 + tid / 16, ek = b.z;
  double *q = uq + ((int64_t)(b.x + gridDim.x * b.y) * G.nez + ek) * 27 * 256 + tid;
  if (ex < 0 || ex >= G.nex || ey < 0 || ey >= G.ney) {
    for (int g = 0; g < 27; g++) q[g * 256] = 0.;
    return;
  }
  double v[8];
  for (int a = 0; a < 8; a++) v[a] = V[node_id(G, ex + (a & 1), ey + ((a >> 1) & 1), ek + (a >> 2))];
  const double cE = (E_elem ? E_elem[cell_id(G, ex, ey, ek)] : E) * (G.hx * G.hy * G.hz);
  for (int gz = 0; gz < 3; gz++)
    for (int gy = 0; gy < 3; gy++)
      for (int gx = 0; gx < 3; gx++) {
        double vg = 0.;
        for (int a = 0; a < 8; a++)
          vg += ((a & 1) ? gP1(gx) : gP0(gx)) * (((a >> 1) & 1) ? gP1(gy) : gP0(gy)) * ((a >> 2) ? gP1(gz) : gP0(gz)) *
                v[a];
        q[((gz * 3 + gy) * 3 + gx) * 256] = cE * gW(gz) * gW(gx) * gW(gy) * (vg * vg + eta);
      }
}


int64_t uq_doubles(const Grid &G) { return (int64_t)((G.nx + 14) / 15) * ((G.ny + 14) / 15) * G.nez * 27 * 256; }
void launch_u_qsetup(const DevProblem &P, double *uq, hipStream_t s) {
  const dim3 g((P.G.nx + 14) / 15, (P.G.ny + 14) / 15, P.G.nez);
  hipLaunchKernelGGL(k_u_qsetup_lds, g, dim3(256), 0, s, P.G, (const double *)P.V, (const double *)P.E_elem, P.E,
                     P.eta, uq);
}

// ---------------------------------------------------------------- diagonal
// Ke[(a,c),(a,c)] = sum_g W s [(lam+mu) (d_c phi_a)^2 + mu |grad phi_a|^2]
struct UDiagOp {
  static constexpr int NF = 1, NC = 3;
  const double *v;
  double *d;
  const double *E_elem;
  const uint32_t *cmask;  // UNILATERAL_NOCOMPRESSION state
  Grid G;
  BcMask bc;
  double E, lam1, mu1, eta, vol;
  __device__ double load(int, int64_t n) const { return v[n]; }
  // diag_{a,c} = sum_g A_g (d_c N_a)^2 + M_g |grad N_a|^2 with M = W s mu and
  // A = M + the spherical weight.  (d_x N_a)^2 = P_j(y)^2 P_k(z)^2 / hx^2 does
  // not depend on the node's x-index i, so the x-term needs the sums of A and M
  // over gx on the 3 x 3 (gy, gz) lines only, contracted with P_j^2 P_k^2; the
  // y- and z-terms alike.
  __device__ void element(int ex, int ey, int ek, const double (&xin)[2][4][1], double (&r)[8][3]) const {
    double Ee = E_elem ? E_elem[cell_id(G, ex, ey, ek)] : E;
    double cE = Ee * vol;
    const uint32_t cm = cmask[cell_id(G, ex, ey, ek)];
    const double kap1 = (lam1 + 2. * mu1 / 3.) * (1. + eta);
    const double i2[3] = {1. / (G.hx * G.hx), 1. / (G.hy * G.hy), 1. / (G.hz * G.hz)};
    double vx[2][2][3];  // v along x on the (j, k) lines
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int gx = 0; gx < 3; gx++) vx[k][j][gx] = gP0(gx) * xin[k][j * 2][0] + gP1(gx) * xin[k][j * 2 + 1][0];
    // [A, M] summed over gx ([gz][gy]), over gy ([gz][gx]), over gz ([gy][gx])
    double Sx[2][3][3] = {}, Sy[2][3][3] = {}, Sz[2][3][3] = {};
#pragma unroll
    for (int gz = 0; gz < 3; gz++)
#pragma unroll
      for (int gy = 0; gy < 3; gy++)
#pragma unroll
        for (int gx = 0; gx < 3; gx++) {
          const double vv = gP0(gz) * (gP0(gy) * vx[0][0][gx] + gP1(gy) * vx[0][1][gx]) +
                            gP1(gz) * (gP0(gy) * vx[1][0][gx] + gP1(gy) * vx[1][1][gx]);
          const double w = cE * gW(gx) * gW(gy) * gW(gz), s = vv * vv + eta;
          // spherical weight: lam s, or kappa (1 + eta) - 2 mu s / 3 at a compressed point
          const double lw = ((cm >> ((gz * 3 + gy) * 3 + gx)) & 1u) ? w * (kap1 - 2. * mu1 * s / 3.) : w * s * lam1;
          const double mw = w * s * mu1, aw = lw + mw;
          Sx[0][gz][gy] += aw;
          Sx[1][gz][gy] += mw;
          Sy[0][gz][gx] += aw;
          Sy[1][gz][gx] += mw;
          Sz[0][gy][gx] += aw;
          Sz[1][gy][gx] += mw;
        }
    // T[q][b][a] = sum over the two remaining directions of S[q] P_a^2 P_b^2
    double Tx[2][2][2], Ty[2][2][2], Tz[2][2][2];
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int b = 0; b < 2; b++)
#pragma unroll
        for (int a = 0; a < 2; a++) {
          double tx = 0., ty = 0., tz = 0.;
#pragma unroll
          for (int u = 0; u < 3; u++) {
            const double pb = b ? gP1(u) : gP0(u);
#pragma unroll
            for (int t = 0; t < 3; t++) {
              const double pa = a ? gP1(t) : gP0(t), w2 = pa * pa * pb * pb;
              tx += Sx[q][u][t] * w2;
              ty += Sy[q][u][t] * w2;
              tz += Sz[q][u][t] * w2;
            }
          }
          Tx[q][b][a] = tx;  // [k][j]
          Ty[q][b][a] = ty;  // [k][i]
          Tz[q][b][a] = tz;  // [j][i]
        }
#pragma unroll
    for (int a = 0; a < 8; a++) {
      const int i = a & 1, j = (a >> 1) & 1, k = a >> 2;
      const double g2 = i2[0] * Tx[1][k][j] + i2[1] * Ty[1][k][i] + i2[2] * Tz[1][j][i];
      r[a][0] += i2[0] * Tx[0][k][j] + g2;
      r[a][1] += i2[1] * Ty[0][k][i] + g2;
      r[a][2] += i2[2] * Tz[0][j][i] + g2;
    }
  }
  __device__ void store(int i, int j, int k, const double (&acc)[3], const double (&)[1]) const {
    int64_t n = node_id(G, i, j, k);
    for (int c = 0; c < 3; c++) d[3 * n + c] = on_dirichlet(G, bc.face[c], bc.vert[c], i, j, k) ? 1. : acc[c];
  }
};

__global__ __launch_bounds__(256) void k_u_diag_uni(UDiagOp op, int OZ) {
  march<double, 16, 16>(op.G, op, OZ, xcd_block());
}

// The same without compression, from the moments of s = v^2 + eta: (d_x phi_a)^2
// = (1 +- y)^2 (1 +- z)^2 / (16 hx^2) in the element's variables, so its integral
// is a sum of moments without x, in modal form: 1, y, z and yz parts.  Bound by
// FP64 issue on large grids, by latency on small ones: 128^3 114 -> 46 us, a
// cube of 32 elements 13 -> 5.7 us.
struct UDiagModOp {
  using T = double;
  static constexpr int NF = 1, NC = 3;
  const double *v;
  double *d;
  const double *E_elem;
  Grid G;
  BcMask bc;
  double E, eta4, lr1;  // 4 eta; (lam + mu) / mu
  double kd[3];         // vol mu / (16 h_d^2), per 144 times a moment
  struct Face {
    double v[4];
  };
  struct Own {};
  using Aux = double;  // E_e
  using Raw = double;
  static __device__ double off() { return 0.; }
  __device__ double load(int, int64_t n) const { return v[n]; }
  __device__ double stage(int, double x) const { return x; }
  template <class RD>
  __device__ void face(const RD &rd, Face &F) const {
#pragma unroll
    for (int q = 0; q < 4; q++) F.v[q] = rd(0, q);
  }
  __device__ Own own(const Face &) const { return Own{}; }
  __device__ double aux(int ex, int ey, int ek, int, int) const {
    return E_elem ? E_elem[cell_id(G, ex, ey, ek)] : E;
  }
  __device__ void element(double Ee, const Face &B, const Face &F, double (&tot)[3][4], double (&carry)[3][4]) const {
    double M[3][3][3], I[3][8], sum[8];  // I: of (d_d phi)^2, by modes
    um_moments<double>(B.v, F.v, Ee, eta4, M);
#pragma unroll
    for (int i = 0; i < 8; i++) sum[i] = 0.;
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const int o1 = d == 0 ? 1 : 0, o2 = d == 2 ? 1 : 2;
      double s[3], o[3];
#pragma unroll
      for (int b = 0; b < 3; b++) {
        auto m = [&](int c) { return d == 0 ? M[0][b][c] : d == 1 ? M[b][0][c] : M[b][c][0]; };
        s[b] = m(0) + m(2);
        o[b] = 2. * m(1);
      }
#pragma unroll
      for (int i = 0; i < 8; i++) I[d][i] = 0.;
      I[d][0] = kd[d] * (s[0] + s[2]);
      I[d][1 << o1] = kd[d] * (2. * s[1]);
      I[d][1 << o2] = kd[d] * (o[0] + o[2]);
      I[d][1 << o1 | 1 << o2] = kd[d] * (2. * o[1]);
#pragma unroll
      for (int i = 0; i < 8; i++) sum[i] += I[d][i];
    }
#pragma unroll
    for (int c = 0; c < 3; c++) {
      double R[8];
#pragma unroll
      for (int i = 0; i < 8; i++) R[i] = sum[i] + lr1 * I[c][i];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        tot[c][q] += R[q] - R[q + 4];
        carry[c][q] = R[q] + R[q + 4];
      }
    }
  }
  __device__ void store(int64_t n, uint32_t fb, const double (&acc)[3], const Own &) const {
#pragma unroll
    for (int c = 0; c < 3; c++) d[3 * n + c] = face_dirichlet(bc.face[c], bc.vert[c], fb) ? 1. : acc[c];
  }
};
template <int W>
__global__ __launch_bounds__(W *W, 2) void k_u_diag(UDiagModOp op, int OZ) {
  march_modal<W, W>(op.G, op, OZ, xcd_block());
}

// ------------------------------------------------------- load vector / residual
// b_{a,c} = sum_g W d_c phi_a [(3lam+2mu) alpha dth s + beta p v]          (thermo-poro)
//         + sum_g W p (d_c v) phi_a                       (crack pressure, optional)
// mode 0: out = b (no BC); mode 1: out = K U - b with ResidualApplyDirichletBC
// Load terms of the residual for one element: at every Gauss point the
// damaged thermal / poroelastic stress tp (times grad N_a) and the crack
// pressure term cp grad(v) (times N_a), both scaled by sgn, added into r.
// The fields are interpolated along x first, and the projection is contracted
// over gx, then gy, then added per gz.
__device__ __forceinline__ void rhs_loads(const double (&X)[2][4][6], double coefalpha, double beta, double eta,
                                          double vol, bool crack, const double (&ih)[3], uint32_t cm, double sgn,
                                          double (&r)[8][3]) {
  double f1[3][2][2][3], dvx[2][2];  // [v, th, p][k][j][gx] interpolated along x; dv/dx on the (j, k) lines
#pragma unroll
  for (int k = 0; k < 2; k++)
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const double *a0 = X[k][j * 2], *a1 = X[k][j * 2 + 1];
#pragma unroll
      for (int f = 0; f < 3; f++)
#pragma unroll
        for (int gx = 0; gx < 3; gx++) f1[f][k][j][gx] = gP0(gx) * a0[3 + f] + gP1(gx) * a1[3 + f];
      dvx[k][j] = (a1[3] - a0[3]) * ih[0];
    }
#pragma unroll
  for (int gz = 0; gz < 3; gz++) {
    double SA[3], SAi[2][3], SB[3][2][3];  // sums over gx: of tp; of tp P_i; of B_c P_i  ([..][gy])
#pragma unroll
    for (int gy = 0; gy < 3; gy++) {
      const double wjk[2][2] = {{gP0(gy) * gP0(gz), gP1(gy) * gP0(gz)}, {gP0(gy) * gP1(gz), gP1(gy) * gP1(gz)}};
      const double gvx = wjk[0][0] * dvx[0][0] + wjk[0][1] * dvx[0][1] + wjk[1][0] * dvx[1][0] + wjk[1][1] * dvx[1][1];
      SA[gy] = 0.;
#pragma unroll
      for (int i = 0; i < 2; i++) {
        SAi[i][gy] = 0.;
#pragma unroll
        for (int c = 0; c < 3; c++) SB[c][i][gy] = 0.;
      }
#pragma unroll
      for (int gx = 0; gx < 3; gx++) {
        double vv = 0., th = 0., pr = 0.;
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
          for (int j = 0; j < 2; j++) {
            vv += wjk[k][j] * f1[0][k][j][gx];
            th += wjk[k][j] * f1[1][k][j][gx];
            pr += wjk[k][j] * f1[2][k][j][gx];
          }
        const double gvy = ih[1] * (gP0(gz) * (f1[0][0][1][gx] - f1[0][0][0][gx]) +
                                    gP1(gz) * (f1[0][1][1][gx] - f1[0][1][0][gx]));
        const double gvz = ih[2] * (gP0(gy) * (f1[0][1][0][gx] - f1[0][0][0][gx]) +
                                    gP1(gy) * (f1[0][1][1][gx] - f1[0][0][1][gx]));
        const double W = vol * gW(gx) * gW(gy) * gW(gz);
        const bool comp = (cm >> ((gz * 3 + gy) * 3 + gx)) & 1u;  // VFMech.c:505-513
        const double tp = sgn * (comp ? W * (coefalpha * th * (1. + eta) + beta * pr)
                                      : W * (coefalpha * th * (vv * vv + eta) + beta * pr * vv));
        const double cp = crack ? sgn * W * pr : 0.;
        const double B[3] = {cp * gvx, cp * gvy, cp * gvz};
        SA[gy] += tp;
        SAi[0][gy] += tp * gP0(gx);
        SAi[1][gy] += tp * gP1(gx);
#pragma unroll
        for (int c = 0; c < 3; c++) {
          SB[c][0][gy] += B[c] * gP0(gx);
          SB[c][1][gy] += B[c] * gP1(gx);
        }
      }
    }
    // corner a = (i, j, k): x-term sx P_j P_k, y-term P_i sy P_k, z-term
    // P_i P_j sz (s = -+1/h), N-term P_i P_j P_k
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const double pz = k ? gP1(gz) : gP0(gz), sz = k ? ih[2] : -ih[2];
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const double sy = j ? ih[1] : -ih[1];
        double TAx = 0., TAy[2] = {0., 0.}, TAz[2] = {0., 0.}, TB[3][2] = {{0., 0.}, {0., 0.}, {0., 0.}};
#pragma unroll
        for (int gy = 0; gy < 3; gy++) {
          const double py = j ? gP1(gy) : gP0(gy);
          TAx += SA[gy] * py;
#pragma unroll
          for (int i = 0; i < 2; i++) {
            TAy[i] += SAi[i][gy];
            TAz[i] += SAi[i][gy] * py;
#pragma unroll
            for (int c = 0; c < 3; c++) TB[c][i] += SB[c][i][gy] * py;
          }
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
          const double sx = i ? ih[0] : -ih[0];
          const int a = (k * 2 + j) * 2 + i;
          r[a][0] += pz * (sx * TAx + TB[0][i]);
          r[a][1] += pz * (sy * TAy[i] + TB[1][i]);
          r[a][2] += sz * TAz[i] + pz * TB[2][i];
        }
      }
    }
  }
}

// residual and loads under UNILATERAL_NOCOMPRESSION in one pass: both follow
// the branch of every Gauss point
struct URhsOp {
  static constexpr int NF = 6, NC = 3;  // u0,u1,u2,v,dth,p
  const double *U, *v, *dth, *p, *BCU;
  double *out;
  const double *E_elem;
  Grid G;
  BcMask bc;
  uint8_t ftype[3][6];   // face types for the residual BC values
  uint8_t vtype[3][8];
  double E, lam1, mu1, eta, vol, alpha, beta;
  int crack, mode;
  __device__ double load(int f, int64_t n) const {
    return f < 3 ? U[3 * n + f] : f == 3 ? v[n] : f == 4 ? dth[n] : p[n];
  }
  __device__ void element(int ex, int ey, int ek, const double (&X)[2][4][6], double (&r)[8][3]) const {
    double Ee = E_elem ? E_elem[cell_id(G, ex, ey, ek)] : E;
    double lam = lam1 * Ee, mu = mu1 * Ee;
    const double ih[3] = {1. / G.hx, 1. / G.hy, 1. / G.hz};
    // the branch of every Gauss point follows U itself (VFMech.c:1566-1615:
    // VF_UResidual evaluates both terms at the iterate)
    double u[8][3];
    for (int a = 0; a < 8; a++)
      for (int c = 0; c < 3; c++) u[a][c] = X[a >> 2][a & 3][c];
    const uint32_t cm = compression_mask(u, ih[0], ih[1], ih[2]);
    if (mode == 1) {
      double Xa[2][4][4];
      for (int k = 0; k < 2; k++)
        for (int q = 0; q < 4; q++)
          for (int f = 0; f < 4; f++) Xa[k][q][f] = X[k][q][f];
      u_elem_apply<double>(Xa, Ee * vol, lam1, mu1, eta, ih[0], ih[1], ih[2], r, cm);
    }
    const double coefalpha = (3. * lam + 2. * mu) * alpha;
    rhs_loads(X, coefalpha, beta, eta, vol, crack != 0, ih, cm, mode == 1 ? -1. : 1., r);
  }
  // value written by ResidualApplyDirichletBC: traversal order X0..Z1 then
  // vertices, later writers win (VFCartFE.c:747-999)
  __device__ void store(int i, int j, int k, const double (&acc)[3], const double (&own)[6]) const {
    int64_t n = node_id(G, i, j, k);
    for (int c = 0; c < 3; c++) {
      double val = acc[c];
      if (mode == 1 && on_dirichlet(G, bc.face[c], bc.vert[c], i, j, k)) {
        int t = 0;
        const bool onf[6] = {i == 0, i == G.nx - 1, j == 0, j == G.ny - 1, k == 0, k == G.nz - 1};
        for (int f = 0; f < 6; f++)
          if (ftype[c][f] && onf[f]) t = ftype[c][f];
        int ix = (i == 0) ? 0 : (i == G.nx - 1) ? 1 : -1;
        int iy = (j == 0) ? 0 : (j == G.ny - 1) ? 1 : -1;
        int iz = (k == 0) ? 0 : (k == G.nz - 1) ? 1 : -1;
        if (ix >= 0 && iy >= 0 && iz >= 0 && vtype[c][ix + 2 * iy + 4 * iz]) t = vtype[c][ix + 2 * iy + 4 * iz];
        double u = own[c];
        val = t == 3 ? u - BCU[3 * n + c] : t == 2 ? u - 1. : u;
      }
      out[3 * n + c] = val;
    }
  }
};

// The load vector alone (UNILATERAL_NONE: the loads do not depend on U):
// mode 0 stores b; mode 1 finishes the residual F = K U - b over an output
// that already holds K U (the FP64 apply), and writes the Dirichlet rows'
// ResidualApplyDirichletBC values from U (read there only); mode 2 stores b
// with the Dirichlet rows' targets instead, so that F(U) = A U - b for the
// MatShell operator A.
//
// With R the modal duals of the nodal loads (x mono = the monomial of a mode):
//   thermo-poro (VFMech.c:386-447): R_d,i = vol / (4 h_d) <T mono_i / x_d> for
//     the modes i with variable d, T = (3 lam + 2 mu) alpha dth (v^2 + eta) +
//     beta p v: 7 moments of T, summed over its 27 Gauss points;
//   crack pressure (VFMech.c:533-589): R_d,i = vol / 8 <p (d_d v) mono_i>, in
//     closed form (d_d v does not depend on x_d).
// Bound by issue, about 500 FP64 operations per element against 1300 of two
// walks over the Gauss points into the corners: 101 x 88 x 95 in 45 us (first
// touch), 72 us so; in small grids apply + loads 27 us against 47 us of both
// in one spilling kernel.
struct ULoadsOp {
  using T = double;
  static constexpr int NF = 3, NC = 3;  // v, dth, p
  const double *U, *v, *dth, *p, *BCU;
  double *out;
  const double *E_elem;
  Grid G;
  BcMask bc;
  uint8_t ftype[3][6];
  uint8_t vtype[3][8];
  double E, ca, beta, eta64;  // (3 lam + 2 mu) alpha / 8 for E = 1; eta of 8 v
  double kt[3][3], kp[3];     // per component: thermo-poro (by odd powers), crack pressure
  int crack, mode;
  struct Face {
    double v[5], t[4], p[4];  // v: first corner, then s, x, y, w of the differences to it
  };
  struct Own {};
  using Aux = double;  // E_e
  using Raw = double;
  static __device__ double off() { return 0.; }
  __device__ double load(int f, int64_t n) const { return f == 0 ? v[n] : f == 1 ? dth[n] : p[n]; }
  __device__ double stage(int, double x) const { return x; }
  template <class RD>
  __device__ void face(const RD &rd, Face &F) const {
    {
      const double x0 = rd(0, 0), b = rd(0, 1) - x0, e = rd(0, 2) - x0, d = rd(0, 3) - x0, t = d - e;
      F.v[0] = x0;
      F.v[2] = t + b;
      F.v[4] = t - b;
      F.v[3] = 2. * d - F.v[2];
      F.v[1] = 2. * d - F.v[4];
    }
#pragma unroll
    for (int f = 1; f < 3; f++) {
      double(&o)[4] = f == 1 ? F.t : F.p;
      const double x0 = rd(f, 0), x1 = rd(f, 1), x2 = rd(f, 2), x3 = rd(f, 3);
      const double s0 = x0 + x1, s1 = x2 + x3, d0 = x1 - x0, d1 = x3 - x2;
      o[0] = s0 + s1;
      o[1] = d0 + d1;
      o[2] = s1 - s0;
      o[3] = d1 - d0;
    }
  }
  __device__ Own own(const Face &) const { return Own{}; }
  __device__ double aux(int ex, int ey, int ek, int, int) const {
    return E_elem ? E_elem[cell_id(G, ex, ey, ek)] : E;
  }
  __device__ void element(double Ee, const Face &B, const Face &F, double (&tot)[3][4], double (&carry)[3][4]) const {
    double V[8], Th[8], Pm[8], m[8];
    V[0] = 4. * (F.v[0] + B.v[0]) + (F.v[1] + B.v[1]);
    V[4] = 4. * (F.v[0] - B.v[0]) + (F.v[1] - B.v[1]);
#pragma unroll
    for (int q = 1; q < 4; q++) {
      V[q] = F.v[q + 1] + B.v[q + 1];
      V[q + 4] = F.v[q + 1] - B.v[q + 1];
    }
    const double ce = ca * Ee;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      Th[q] = ce * (F.t[q] + B.t[q]);
      Th[q + 4] = ce * (F.t[q] - B.t[q]);
      Pm[q] = F.p[q] + B.p[q];
      Pm[q + 4] = F.p[q] - B.p[q];
    }
#pragma unroll
    for (int i = 0; i < 8; i++) m[i] = 0.;  // moments of 64 T; the common weight is in kt
#pragma unroll
    for (int gz = 0; gz < 3; gz++) {
      double f[3][4], L[4] = {0., 0., 0., 0.};
#pragma unroll
      for (int q = 0; q < 4; q++) {
        f[0][q] = at_gauss(gz, V[q], V[q + 4]);
        f[1][q] = at_gauss(gz, Th[q], Th[q + 4]);
        f[2][q] = beta * at_gauss(gz, Pm[q], Pm[q + 4]);
      }
#pragma unroll
      for (int gy = 0; gy < 3; gy++) {
        double t[3], r[3][2];
#pragma unroll
        for (int c = 0; c < 3; c++) {
          r[c][0] = at_gauss(gy, f[c][0], f[c][2]);
          r[c][1] = at_gauss(gy, f[c][1], f[c][3]);
        }
#pragma unroll
        for (int gx = 0; gx < 3; gx++) {
          const double vg = at_gauss(gx, r[0][0], r[0][1]);
          t[gx] = at_gauss(gx, r[1][0], r[1][1]) * (vg * vg + eta64) + at_gauss(gx, r[2][0], r[2][1]) * vg;
        }
        const double s = (t[0] + t[2]) + 1.6 * t[1], o = t[2] - t[0];  // weights 5 : 8 : 5
        L[0] += gy == 1 ? 1.6 * s : s;
        L[1] += gy == 1 ? 1.6 * o : o;
        if (gy != 1) {
          L[2] += gy ? s : -s;
          L[3] += gy ? o : -o;
        }
      }
#pragma unroll
      for (int q = 0; q < 4; q++) {
        m[q] += gz == 1 ? 1.6 * L[q] : L[q];
        if (gz != 1 && q < 3) m[q + 4] += gz ? L[q] : -L[q];
      }
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
      double R[8];
#pragma unroll
      for (int i = 0; i < 8; i++)
        R[i] = um_pow(i, d) ? kt[d][__builtin_popcount(i) - 1] * m[i & ~(1 << d)] : 0.;
      if (crack) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
          double p2[2][2], v2[2][2], M[2][2];
#pragma unroll
          for (int q = 0; q < 4; q++) {
            p2[q & 1][q >> 1] = Pm[modal_at(d, t, q & 1, q >> 1)];
            v2[q & 1][q >> 1] = kp[d] * V[modal_at(d, 1, q & 1, q >> 1)];
          }
          bilinear_moments(p2, v2, M);
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const int o = t + (q & 1) + (q >> 1);
            R[modal_at(d, t, q & 1, q >> 1)] +=
                (o == 0 ? 1. : o == 1 ? 1. / 3. : o == 2 ? 1. / 9. : 1. / 27.) * M[q & 1][q >> 1];
          }
        }
      }
#pragma unroll
      for (int q = 0; q < 4; q++) {
        tot[d][q] += R[q] - R[q + 4];
        carry[d][q] = R[q] + R[q + 4];
      }
    }
  }
  struct OwnKU {
    double f[3];
  };
  __device__ OwnKU own_load(int64_t n) const {
    OwnKU o{};
    if (mode == 1)
#pragma unroll
      for (int c = 0; c < 3; c++) o.f[c] = out[3 * n + c];
    return o;
  }
  __device__ void store(int64_t n, uint32_t fb, const double (&acc)[3], const Own &, const OwnKU &o) const {
    double val[3];
#pragma unroll
    for (int c = 0; c < 3; c++) val[c] = o.f[c] + acc[c];  // mode 1: K U - b
    if (mode != 0 && fb) {
#pragma unroll
      for (int c = 0; c < 3; c++)
        if (face_dirichlet(bc.face[c], bc.vert[c], fb)) {
          const double w = dirichlet_value(fb, c, n);
          val[c] = mode == 1 ? U[3 * n + c] - w : w;
        }
    }
#pragma unroll
    for (int c = 0; c < 3; c++) out[3 * n + c] = val[c];
  }
  // ResidualApplyDirichletBC's target on a Dirichlet row: BCU (type 3), 1 (type 2), else 0
  __device__ double dirichlet_value(uint32_t fb, int c, int64_t n) const {
    int t = 0;
    for (int f = 0; f < 6; f++)
      if (ftype[c][f] && (fb >> f & 1u)) t = ftype[c][f];
    const int q = face_vertex(fb);
    if (q >= 0 && vtype[c][q]) t = vtype[c][q];
    return t == 3 ? BCU[3 * n + c] : t == 2 ? 1. : 0.;
  }
};
template <int W>
__global__ __launch_bounds__(W *W, 2) void k_u_loads(ULoadsOp op, int OZ) {
  march_modal<W, W>(op.G, op, OZ, xcd_block());
}

__global__ __launch_bounds__(256) void k_u_rhs(URhsOp op, int OZ) {
  march<double, 16, 16>(op.G, op, OZ, xcd_block());
}

// ------------------------------------------------------------ host launchers
static dim3 march_grid(const Grid &G, int TX, int TY, int OZ) {
  return dim3((G.nx + TX - 2) / (TX - 1), (G.ny + TY - 2) / (TY - 1), (G.nz + OZ - 1) / OZ);
}

// z-chunk length of the marching tiles: every chunk recomputes one element
// layer below it, so long chunks waste less; the grid should still fill every
// workgroup slot of the device.  Minimise rounds * (layers per workgroup),
// rounds = ceil(workgroups / resident slots).
// One plane per chunk where that still fits the device at once: two layers of
// latency instead of three (17 x 12 x 20 elements FP64 20.3 -> 18.2 us, a solve
// of 32^3 1.69 -> 1.60 ms).
int choose_oz(const Grid &G, int tiles_xy, int slots) {
  if (slots < 1) slots = 256;
  int best = G.nz;
  double best_cost = 1e300;
  for (int oz = 1; oz <= G.nz; oz++) {
    int chunks = (G.nz + oz - 1) / oz;
    if (oz > 1 && (G.nz + oz - 2) / (oz - 1) == chunks) continue;  // same chunk count, shorter is free
    int64_t wg = (int64_t)tiles_xy * chunks;
    double rounds = (double)((wg + slots - 1) / slots);
    double cost = rounds * (oz + 1);
    if (cost < best_cost - 1e-9) { best_cost = cost; best = oz; }
  }
  return best;
}

// resident workgroups of a kernel on the whole device (occupancy x CUs)
int device_slots_of(const void *kernel, int threads) {
  static int cus = 0;
  if (!cus) {
    int dev = 0;
    hipGetDevice(&dev);
    hipDeviceProp_t pr;
    cus = hipGetDeviceProperties(&pr, dev) == hipSuccess ? pr.multiProcessorCount : 256;
  }
  int per = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, threads, 0) != hipSuccess || per < 1) per = 1;
  return per * cus;
}
template <typename K>
static int device_slots(K kernel, int threads) {
  return device_slots_of((const void *)kernel, threads);
}

// FP32 grids of 16-64 nodes in x (coarse multigrid levels) march 8 x 8 tiles
// of 7 x 7 owned nodes: more, shorter workgroups, and no row of 15-node tiles whose
// last owns a node or two.  Apply in 16 x 16 and 8 x 8 tiles, cubes of nodes: 9
// 6.1 and 6.6 us, 15 6.3 and 6.0, 17 11.6 and 6.1, 22 6.3 and 7.0, 25 6.3 and 6.3, 31
// 10.8 and 6.3, 33 7.8 and 6.4, 49 9.9 and 9.7, 57 9.9 and 12.8, 64 and 65 15.2 and
// 15.0, 129 52.3 and 56.9; 17 x 513 x 513 153 and 118, 33 x 257 x 257 64 and 58,
// 129 x 129 x 9 9.4 and 9.9.  Outside the range the two are within 8 % (the
// narrowest, 129 x 17 x 17 and 257 x 9 x 9: 7.5 and 6.3, 6.7 and 6.2).
constexpr int SMALL_NX_LO = 16, SMALL_NX_HI = 64;
// FP64 grids whose 8 x 8 tiles all run at once in chunks of one node plane take
// them: the one-wavefront workgroups start and synchronise faster (cubes of 16
// elements 11.1 -> 6.2 us, 32 9.0 -> 6.7, 40 equal; 44 and 56, which no longer
// fit, 9.3 -> 11.9 and 12.8 -> 15.4 us)
static bool small_fp64(const Grid &G);
template <typename T>
static void launch_u_apply_uni(const DevProblem &P, const T *x, T *y, const T *v, hipStream_t s) {
  UApplyUniOp<T> op;
  op.x = x; op.y = y; op.v = v;
  op.E_elem = P.E_elem;
  op.cmask = P.cmask;
  op.G = P.G; op.bc = P.bcU;
  op.E = T(P.E); op.lam1 = T(P.lam1); op.mu1 = T(P.mu1); op.eta = T(P.eta);
  op.vol = T(P.G.hx * P.G.hy * P.G.hz);
  op.ihx = T(1. / P.G.hx); op.ihy = T(1. / P.G.hy); op.ihz = T(1. / P.G.hz);
  const int tiles = ((P.G.nx + 14) / 15) * ((P.G.ny + 14) / 15);
  static int slots = device_slots(k_u_apply_uni<T, 16, 16>, 256);
  const int OZ = choose_oz(P.G, tiles, slots);
  hipLaunchKernelGGL((k_u_apply_uni<T, 16, 16>), march_grid(P.G, 16, 16, OZ), dim3(256), 0, s, op, OZ);
}
template <typename T, int W, bool UNIT, bool CUBIC>
static void launch_u_apply_c(const UModRec<T> &r, hipStream_t s) {
  UModOp<T, UNIT, CUBIC> op;
  static_cast<UModRec<T> &>(op) = r;
  const Grid &G = r.G;
  static int slots = device_slots(k_u_apply<T, W, W, UNIT, CUBIC>, W * W);
  const int OZ = choose_oz(G, ((G.nx + W - 2) / (W - 1)) * ((G.ny + W - 2) / (W - 1)), slots);
  hipLaunchKernelGGL((k_u_apply<T, W, W, UNIT, CUBIC>), march_grid(G, W, W, OZ), dim3(W * W), 0, s, op, OZ);
}
template <typename T, int W, bool UNIT>
static void launch_u_apply_w(const DevProblem &P, const T *x, T *y, hipStream_t s) {
  UModRec<T> r;
  umod_fill<T>(r, P, x, y);
  r.m.cubic ? launch_u_apply_c<T, W, UNIT, true>(r, s) : launch_u_apply_c<T, W, UNIT, false>(r, s);
}

template <typename T>
static void launch_u_apply_t(const DevProblem &P, const T *x, T *y, const T *v, hipStream_t s) {
  if (P.unilateral) {
    launch_u_apply_uni<T>(P, x, y, v, s);
    return;
  }
  if constexpr (sizeof(T) == 8) {
    if (P.uq) {
      UApplyLdsqOp<false> q;
      q.x = (const double *)x; q.y = (double *)y; q.part = nullptr; q.uq = P.uq;
      q.G = P.G; q.bc = P.bcU; q.lam1 = P.lam1; q.mu1 = P.mu1;
      q.ihx = 1. / P.G.hx; q.ihy = 1. / P.G.hy; q.ihz = 1. / P.G.hz;
      const int tiles = ((P.G.nx + 14) / 15) * ((P.G.ny + 14) / 15);
      static int lqslots = device_slots(k_u_apply_ldsq, 256);
      const int OZ = choose_oz(P.G, tiles, lqslots);
      hipLaunchKernelGGL(k_u_apply_ldsq, march_grid(P.G, 16, 16, OZ), dim3(256), 0, s, q, OZ);
      return;
    }
    small_fp64(P.G) ? launch_u_apply_w<T, 8, false>(P, x, y, s) : launch_u_apply_w<T, 16, false>(P, x, y, s);
  } else {
    const bool small = P.G.nx >= SMALL_NX_LO && P.G.nx <= SMALL_NX_HI;
    if (P.unit) small ? launch_u_apply_w<T, 8, true>(P, x, y, s) : launch_u_apply_w<T, 16, true>(P, x, y, s);
    else small ? launch_u_apply_w<T, 8, false>(P, x, y, s) : launch_u_apply_w<T, 16, false>(P, x, y, s);
  }
}

static bool small_fp64(const Grid &G) {
  static int slots = device_slots(k_u_apply<double, 8, 8, false, false>, 64);
  return (int64_t)((G.nx + 6) / 7) * ((G.ny + 6) / 7) * G.nz <= slots;
}

// per element: the Gauss points where tr(eps(U)) < 0
__global__ void k_u_cmask(Grid G, const double *__restrict__ U, uint32_t *__restrict__ cmask) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)G.nex * G.ney * G.nez) return;
  const int ei = (int)(e % G.nex), ej = (int)((e / G.nex) % G.ney), ek = (int)(e / ((int64_t)G.nex * G.ney));
  double u[8][3];
  for (int a = 0; a < 8; a++) {
    const int64_t n = node_id(G, ei + (a & 1), ej + ((a >> 1) & 1), ek + (a >> 2));
    for (int c = 0; c < 3; c++) u[a][c] = U[3 * n + c];
  }
  cmask[e] = compression_mask(u, 1. / G.hx, 1. / G.hy, 1. / G.hz);
}

void launch_u_cmask(const DevProblem &P, const double *U, hipStream_t s) {
  hipLaunchKernelGGL(k_u_cmask, dim3((unsigned)((P.ne + 255) / 256)), dim3(256), 0, s, P.G, U, P.cmask);
}

// one apply record of the batched / engine applies
template <typename T>
struct BApply {
  UModRec<T> op;
  int OZ;
};
// the kernel's op from a record
template <class Op>
__device__ __forceinline__ Op op_of(const typename Op::Record &r) {
  Op o;
  static_cast<typename Op::Record &>(o) = r;
  return o;
}

// Chebyshev-Jacobi solve of a small FP32 level from x = 0 in one workgroup
// (the coarsest multigrid level, at most 8 elements per direction).  A thread
// owns one element (its modulus and place are read once) and up to MGC_Q nodes,
// whose b, D^-1, x and direction stay in its registers; only the iterate and the
// element forces go through LDS, component by component so that consecutive
// lanes touch consecutive words.  A step is an element pass and a node pass that
// adds each node's eight element forces in a fixed order (x-pairs, then y-pairs,
// the lower element layer before the upper); the step itself is
// mg_cheb_entry's.  LDS is laid out for 8^3 elements whatever the level has, the
// forces with a border of elements that stay zero: every address is a thread's
// base plus a constant (a table of the forces' places, formed with divisions by
// the level's extents, cost a quarter of the time).  Latency-bound on one CU:
// 9^3 nodes 15 -> 11.7 us.
constexpr int MGC_E = 8, MGC_N = MGC_E + 1, MGC_P = MGC_E + 2;  // elements, nodes, bordered elements per direction
constexpr int MGC_T = MGC_E * MGC_E * MGC_E, MGC_NN = MGC_N * MGC_N * MGC_N, MGC_NP = MGC_P * MGC_P * MGC_P;
constexpr int MGC_Q = (MGC_NN + MGC_T - 1) / MGC_T;
struct MgcLds {
  float x[3 * MGC_NN];
  alignas(16) float r[24 * MGC_NP];  // [corner * 3 + component][bordered element]
};

// coef(i): the step's coefficients {c1, c2}
template <bool UNIT, bool CUBIC, class Coef>
__device__ __forceinline__ void mg_coarse_cheb_body(MgcLds &S, const UModRec<float> &rec, const float *__restrict__ b,
                                                    const float *__restrict__ dinv, float *__restrict__ xout,
                                                    int steps, const Coef &coef) {
  const Grid &G = rec.G;
  const int tid = threadIdx.x;
  // the nodes tid + q MGC_T of a 9^3 grid
  float eb[MGC_Q][3], ed[MGC_Q][3], xe[MGC_Q][3], dir[MGC_Q][3];
  uint32_t fixed[MGC_Q];  // components on Dirichlet rows
  int node[MGC_Q];        // of the level, -1: none
  int src[MGC_Q];         // bordered element above the node
#pragma unroll
  for (int q = 0; q < MGC_Q; q++) {
    const int t = tid + q * MGC_T, i = t % MGC_N, j = t / MGC_N % MGC_N, k = t / (MGC_N * MGC_N);
    const bool in = t < MGC_NN && i < G.nx && j < G.ny && k < G.nz;
    node[q] = in ? i + G.nx * (j + G.ny * k) : -1;
    src[q] = in ? (i + 1) + MGC_P * ((j + 1) + MGC_P * (k + 1)) : MGC_NP - 1;
    fixed[q] = 0u;
    const uint32_t fb = face_bits_xy(G, i, j) | (k == 0 ? 16u : 0u) | (k == G.nz - 1 ? 32u : 0u);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      eb[q][c] = in ? b[3 * node[q] + c] : 0.f;
      ed[q][c] = in ? dinv[3 * node[q] + c] : 0.f;
      xe[q][c] = dir[q][c] = 0.f;
      if (face_dirichlet(rec.bc.face[c], rec.bc.vert[c], fb)) fixed[q] |= 1u << c;
    }
  }
  // the thread's element
  const int ex = tid % MGC_E, ey = tid / MGC_E % MGC_E, ez = tid / (MGC_E * MGC_E);
  const bool el = ex < G.nex && ey < G.ney && ez < G.nez;
  const int n0 = ex + MGC_N * (ey + MGC_N * ez), e0 = (ex + 1) + MGC_P * ((ey + 1) + MGC_P * (ez + 1));
  float E = 0.f, vb[4] = {}, vt[4] = {};
  if (el) {
    E = rec.E_elem ? (float)rec.E_elem[cell_id(G, ex, ey, ez)] : rec.E;
    if constexpr (!UNIT)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        vb[q] = rec.v[node_id(G, ex + (q & 1), ey + (q >> 1), ez)];
        vt[q] = rec.v[node_id(G, ex + (q & 1), ey + (q >> 1), ez + 1)];
      }
  }
  for (int i = tid; i < 24 * MGC_NP / 4; i += MGC_T) ((float4 *)S.r)[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int i = 0; i < steps; i++) {
    const BmgCoef cf = coef(i);
    if (i > 0) {
#pragma unroll
      for (int q = 0; q < MGC_Q; q++)
        if (tid + q * MGC_T < MGC_NN)
#pragma unroll
          for (int c = 0; c < 3; c++) S.x[c * MGC_NN + tid + q * MGC_T] = xe[q][c];
      __syncthreads();
      if (el) {
        UFace<float> fb, ft;
        float t[2][3][4] = {};
#pragma unroll
        for (int c = 0; c < 3; c++) {
          const float *xb = S.x + c * MGC_NN + n0, *xt = xb + MGC_N * MGC_N;
          uface_set<float>(fb, c, xb[0], xb[1], xb[MGC_N], xb[MGC_N + 1]);
          uface_set<float>(ft, c, xt[0], xt[1], xt[MGC_N], xt[MGC_N + 1]);
        }
        um_layer<float, UNIT, CUBIC>(fb, ft, vb, vt, E, rec.m, t[0], t[1]);
#pragma unroll
        for (int kz = 0; kz < 2; kz++)
#pragma unroll
          for (int c = 0; c < 3; c++) {
            const float(&u)[4] = t[kz][c];
            const float p0 = u[0] - u[1], p1 = u[0] + u[1], f0 = u[2] - u[3], f1 = u[2] + u[3];
            float *o = S.r + (kz * 12 + c) * MGC_NP + e0;
            o[0] = p0 - f0;
            o[3 * MGC_NP] = p1 - f1;
            o[6 * MGC_NP] = p0 + f0;
            o[9 * MGC_NP] = p1 + f1;
          }
      }
      __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < MGC_Q; q++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
        float res = eb[q][c];
        if (i > 0) {
          // corner a = 4 K + 2 J + I of the element below by (I, J, K): the layer below (K = 1), then the layer above
          const float *s = S.r + c * MGC_NP + src[q];
          auto at = [&](int a) { return s[a * 3 * MGC_NP - ((a & 1) + MGC_P * ((a >> 1 & 1) + MGC_P * (a >> 2)))]; };
          const float lo = (at(7) + at(6)) + (at(5) + at(4));
          const float y = lo + ((at(3) + at(2)) + (at(1) + at(0)));
          res -= fixed[q] >> c & 1u ? xe[q][c] : y;
        }
        dir[q][c] = (i > 0 ? cf.c1 * dir[q][c] : 0.f) + cf.c2 * ed[q][c] * res;
        xe[q][c] += dir[q][c];
      }
  }
#pragma unroll
  for (int q = 0; q < MGC_Q; q++)
    if (node[q] >= 0)
#pragma unroll
      for (int c = 0; c < 3; c++) xout[3 * node[q] + c] = xe[q][c];
}

template <bool CUBIC>
__global__ __launch_bounds__(MGC_T) void k_mg_coarse_cheb(UModRec<float> rec, const float *__restrict__ b,
                                                          const float *__restrict__ dinv, float *__restrict__ xout,
                                                          MgChebCoefs cc) {
  __shared__ MgcLds S;
  mg_coarse_cheb_body<true, CUBIC>(S, rec, b, dinv, xout, cc.k, [&](int i) { return BmgCoef{cc.c1[i], cc.c2[i]}; });
}

// the batched form: one workgroup per listed member (COARSE: at the level its
// entry names; else level 0, its first chunk), the member's level operator,
// vectors and coarsest-level coefficients from the engine's tables
template <bool COARSE>
__global__ __launch_bounds__(MGC_T) void k_bmg_coarse_cheb(const BmgVec *__restrict__ lvt,
                                                           const BmgChunk *__restrict__ ch, const int *__restrict__ dn,
                                                           const BmgCoef *__restrict__ coef,
                                                           const double *__restrict__ flags, int fstride) {
  if ((int)blockIdx.x >= *dn) return;
  const BmgChunk c = ch[blockIdx.x];
  if ((!COARSE && c.start != 0) || flags[(int64_t)c.p * fstride] == 0.) return;  // uniform in the workgroup
  const int level = COARSE ? (int)c.start : 0;
  const BmgVec &v = lvt[c.p * BML + level];
  const BmgCoef *__restrict__ cf = coef + ((c.p * BML + level) * 2 + 1) * BMK;
  __shared__ MgcLds S;
  const UModRec<float> &rec = ((const BApply<float> *)v.op)->op;
  auto co = [&](int i) { return cf[i]; };
  if (rec.m.cubic) mg_coarse_cheb_body<COARSE, true>(S, rec, v.b, v.dinv, v.x, MG_COARSE_DEG, co);  // uniform
  else mg_coarse_cheb_body<COARSE, false>(S, rec, v.b, v.dinv, v.x, MG_COARSE_DEG, co);
}

bool mg_coarse_fits(const DevProblem &P) {
  return !P.unilateral && P.G.nex <= MGC_E && P.G.ney <= MGC_E && P.G.nez <= MGC_E;
}

void launch_mg_coarse_cheb(const DevProblem &P, const float *b, const float *dinv, float *x, const MgChebCoefs &cc,
                           hipStream_t s) {
  UModRec<float> rec;
  umod_fill<float>(rec, P, nullptr, nullptr);
  auto go = [&](auto k) { hipLaunchKernelGGL(k, dim3(1), dim3(MGC_T), 0, s, rec, b, dinv, x, cc); };
  rec.m.cubic ? go(k_mg_coarse_cheb<true>) : go(k_mg_coarse_cheb<false>);
}

void launch_bmg_coarse_cheb(const BmgVec *lvt, int coarse, const BmgChunk *ch, const int *dn, int grid,
                            const BmgCoef *coef, const double *flags, int fstride, hipStream_t s) {
  if (grid <= 0) return;
  auto go = [&](auto k) { hipLaunchKernelGGL(k, dim3(grid), dim3(MGC_T), 0, s, lvt, ch, dn, coef, flags, fstride); };
  coarse ? go(k_bmg_coarse_cheb<true>) : go(k_bmg_coarse_cheb<false>);
}

void launch_u_apply(const DevProblem &P, const double *x, double *y, hipStream_t s) {
  launch_u_apply_t<double>(P, x, y, P.V, s);
}

template <int W, bool CUBIC>
static int launch_u_apply_dot_c(const UModRec<double> &r, double *part, int max_part, hipStream_t s) {
  UApplyDotOp<CUBIC> op;
  static_cast<UModRec<double> &>(op) = r;
  op.part = part;
  const Grid &G = r.G;
  static int slots = device_slots(k_u_apply_dot<W, CUBIC>, W * W);
  const int OZ = choose_oz(G, ((G.nx + W - 2) / (W - 1)) * ((G.ny + W - 2) / (W - 1)), slots);
  const dim3 g = march_grid(G, W, W, OZ);
  const int64_t nwg = (int64_t)g.x * g.y * g.z;
  if (nwg > max_part) return 0;
  hipLaunchKernelGGL((k_u_apply_dot<W, CUBIC>), g, dim3(W * W), 0, s, op, OZ);
  return (int)nwg;
}
int launch_u_apply_dot(const DevProblem &P, const double *x, double *y, double *part, int max_part, hipStream_t s) {
  if (P.unilateral) return 0;
  if (P.uq) {
    UApplyLdsqDotOp q;
    q.x = x; q.y = y; q.part = part; q.uq = P.uq;
    q.G = P.G; q.bc = P.bcU; q.lam1 = P.lam1; q.mu1 = P.mu1;
    q.ihx = 1. / P.G.hx; q.ihy = 1. / P.G.hy; q.ihz = 1. / P.G.hz;
    static int lqslots = device_slots(k_u_apply_ldsq_dot, 256);
    const int tiles = ((P.G.nx + 14) / 15) * ((P.G.ny + 14) / 15);
    const int OZ = choose_oz(P.G, tiles, lqslots);
    const dim3 g = march_grid(P.G, 16, 16, OZ);
    const int64_t nwg = (int64_t)g.x * g.y * g.z;
    if (nwg > max_part) return 0;
    hipLaunchKernelGGL(k_u_apply_ldsq_dot, g, dim3(256), 0, s, q, OZ);
    return (int)nwg;
  }
  UModRec<double> r;
  umod_fill<double>(r, P, x, y);
  if (small_fp64(P.G))
    return r.m.cubic ? launch_u_apply_dot_c<8, true>(r, part, max_part, s)
                     : launch_u_apply_dot_c<8, false>(r, part, max_part, s);
  return r.m.cubic ? launch_u_apply_dot_c<16, true>(r, part, max_part, s)
                   : launch_u_apply_dot_c<16, false>(r, part, max_part, s);
}
void launch_u_apply_f32(const DevProblem &P, const float *x, float *y, hipStream_t s) {
  launch_u_apply_t<float>(P, x, y, P.V32, s);
}

static void mg_op_fill(UMgRec &op, const DevProblem &P, const float *b, const float *dinv, float c2) {
  umod_fill<float>(op, P, nullptr, nullptr);
  op.b = b; op.dinv = dinv; op.c2 = c2;
  op.xo = nullptr; op.ro = nullptr; op.r64 = nullptr; op.part = nullptr;
}
// launches 8 x 8 or 16 x 16 tiles by the grid's x extent; returns the workgroup
// count, or 0 without launching when it would exceed max_wg
template <class Op, int W>
static int mg_launch_w(const DevProblem &P, const Op &op, hipStream_t s, int64_t max_wg) {
  static int slots = device_slots(k_u_mg<Op, W, W>, W * W);
  const int OZ = choose_oz(P.G, ((P.G.nx + W - 2) / (W - 1)) * ((P.G.ny + W - 2) / (W - 1)), slots);
  const dim3 g = march_grid(P.G, W, W, OZ);
  const int64_t nwg = (int64_t)g.x * g.y * g.z;
  if (nwg > max_wg) return 0;
  hipLaunchKernelGGL((k_u_mg<Op, W, W>), g, dim3(W * W), 0, s, op, OZ);
  return (int)nwg;
}
template <class Op>
static int mg_launch(const DevProblem &P, const UMgRec &r, hipStream_t s, int64_t max_wg = INT32_MAX) {
  Op op;
  static_cast<UMgRec &>(op) = r;
  const bool small = P.G.nx >= SMALL_NX_LO && P.G.nx <= SMALL_NX_HI;
  return small ? mg_launch_w<Op, 8>(P, op, s, max_wg) : mg_launch_w<Op, 16>(P, op, s, max_wg);
}
void launch_mg_presmooth(const DevProblem &P, const float *b, const float *dinv, float c2, float *x, float *r,
                         hipStream_t s) {
  UMgRec op;
  mg_op_fill(op, P, b, dinv, c2);
  op.xo = x; op.ro = r;
  if (op.m.cubic) P.unit ? mg_launch<UMgPreOp<true, true>>(P, op, s) : mg_launch<UMgPreOp<false, true>>(P, op, s);
  else P.unit ? mg_launch<UMgPreOp<true>>(P, op, s) : mg_launch<UMgPreOp<false>>(P, op, s);
}
int launch_mg_postsmooth(const DevProblem &P, const float *b, const float *dinv, float c2, const float *x, float *xo,
                         const double *r64, double *part, int max_part, hipStream_t s) {
  UMgRec op;
  mg_op_fill(op, P, b, dinv, c2);
  op.x = x; op.xo = xo; op.r64 = r64; op.part = part;
  if (r64) {
    const int n = op.m.cubic ? mg_launch<UMgPostRzOp<true>>(P, op, s, max_part)
                             : mg_launch<UMgPostRzOp<false>>(P, op, s, max_part);
    if (n) return n;  // else too many workgroups for the partials: the plain form
  }
  if (op.m.cubic)
    P.unit ? mg_launch<UMgPostOp<true, false, true>>(P, op, s) : mg_launch<UMgPostOp<false, false, true>>(P, op, s);
  else P.unit ? mg_launch<UMgPostOp<true, false>>(P, op, s) : mg_launch<UMgPostOp<false, false>>(P, op, s);
  return 0;
}

static void launch_u_diag_uni(const DevProblem &P, double *d, hipStream_t s) {
  UDiagOp op;
  op.v = P.V; op.d = d; op.E_elem = P.E_elem; op.G = P.G; op.bc = P.bcU;
  op.cmask = P.cmask;
  op.E = P.E; op.lam1 = P.lam1; op.mu1 = P.mu1; op.eta = P.eta;
  op.vol = P.G.hx * P.G.hy * P.G.hz;
  const int tiles = ((P.G.nx + 14) / 15) * ((P.G.ny + 14) / 15);
  static int slots = device_slots(k_u_diag_uni, 256);
  const int OZ = choose_oz(P.G, tiles, slots);
  hipLaunchKernelGGL(k_u_diag_uni, march_grid(P.G, 16, 16, OZ), dim3(256), 0, s, op, OZ);
}
template <int W>
static void launch_u_diag_w(const UDiagModOp &op, hipStream_t s) {
  const Grid &G = op.G;
  static int slots = device_slots(k_u_diag<W>, W * W);
  const int OZ = choose_oz(G, ((G.nx + W - 2) / (W - 1)) * ((G.ny + W - 2) / (W - 1)), slots);
  hipLaunchKernelGGL(k_u_diag<W>, march_grid(G, W, W, OZ), dim3(W * W), 0, s, op, OZ);
}
void launch_u_diag(const DevProblem &P, double *d, hipStream_t s) {
  if (P.unilateral) return launch_u_diag_uni(P, d, s);
  UDiagModOp op;
  const Grid &G = P.G;
  op.v = P.V; op.d = d; op.E_elem = P.E_elem; op.G = G; op.bc = P.bcU;
  op.E = P.E; op.eta4 = 4. * P.eta; op.lr1 = (P.lam1 + P.mu1) / P.mu1;
  const double h[3] = {G.hx, G.hy, G.hz};
  for (int k = 0; k < 3; k++) op.kd[k] = h[0] * h[1] * h[2] * P.mu1 / (16. * 144. * h[k] * h[k]);
  small_fp64(G) ? launch_u_diag_w<8>(op, s) : launch_u_diag_w<16>(op, s);
}

static void launch_u_rhs_uni(const DevProblem &P, const double *U, const double *BCU, double *out, int mode,
                             hipStream_t s) {
  URhsOp op;
  op.U = U ? U : P.zero3; op.v = P.V; op.dth = P.dth; op.p = P.p; op.BCU = BCU;
  op.out = out; op.E_elem = P.E_elem; op.G = P.G; op.bc = P.bcU;
  for (int c = 0; c < 3; c++) {
    for (int f = 0; f < 6; f++) op.ftype[c][f] = (uint8_t)P.hbcU[c].face[f];
    for (int v = 0; v < 8; v++) op.vtype[c][v] = (uint8_t)P.hbcU[c].vertex[v];
  }
  op.E = P.E; op.lam1 = P.lam1; op.mu1 = P.mu1; op.eta = P.eta;
  op.vol = P.G.hx * P.G.hy * P.G.hz; op.alpha = P.alpha; op.beta = P.beta;
  op.crack = P.hasCrackPressure; op.mode = mode;
  int tiles = ((P.G.nx + 14) / 15) * ((P.G.ny + 14) / 15);
  static int slots = device_slots(k_u_rhs, 256);
  int OZ = choose_oz(P.G, tiles, slots);
  hipLaunchKernelGGL(k_u_rhs, march_grid(P.G, 16, 16, OZ), dim3(256), 0, s, op, OZ);
}

template <int W>
static void launch_u_loads_w(const ULoadsOp &op, hipStream_t s) {
  const Grid &G = op.G;
  static int slots = device_slots(k_u_loads<W>, W * W);
  const int OZ = choose_oz(G, ((G.nx + W - 2) / (W - 1)) * ((G.ny + W - 2) / (W - 1)), slots);
  hipLaunchKernelGGL(k_u_loads<W>, march_grid(G, W, W, OZ), dim3(W * W), 0, s, op, OZ);
}
void launch_u_rhs(const DevProblem &P, const double *U, const double *BCU, double *out, int mode,
                  hipStream_t s) {
  if (P.unilateral) {  // (mode 2 is not used with NOCOMPRESSION: its load depends on U)
    launch_u_rhs_uni(P, U, BCU, out, mode, s);
    return;
  }
  // UNILATERAL_NONE: K U by the FP64 apply, then the loads
  if (mode == 1) launch_u_apply(P, U ? U : P.zero3, out, s);
  ULoadsOp op;
  op.U = U ? U : P.zero3; op.v = P.V; op.dth = P.dth; op.p = P.p; op.BCU = BCU;
  op.out = out; op.E_elem = P.E_elem; op.G = P.G; op.bc = P.bcU;
  for (int c = 0; c < 3; c++) {
    for (int f = 0; f < 6; f++) op.ftype[c][f] = (uint8_t)P.hbcU[c].face[f];
    for (int v = 0; v < 8; v++) op.vtype[c][v] = (uint8_t)P.hbcU[c].vertex[v];
  }
  op.E = P.E; op.beta = P.beta; op.eta64 = 64. * P.eta;
  op.ca = (3. * P.lam1 + 2. * P.mu1) * P.alpha / 8.;
  op.crack = P.hasCrackPressure; op.mode = mode;
  const double h[3] = {P.G.hx, P.G.hy, P.G.hz}, w = (mode == 1 ? -1. : 1.) * h[0] * h[1] * h[2];
  for (int d = 0; d < 3; d++) {
    const double k = w / (4. * 64. * h[d]) * (125. / 5832.);  // (5/18)^3
    op.kt[d][0] = k;
    op.kt[d][1] = k * VFG_SQ35;
    op.kt[d][2] = k * .6;
    op.kp[d] = w / (256. * h[d]);
  }
  small_fp64(P.G) ? launch_u_loads_w<8>(op, s) : launch_u_loads_w<16>(op, s);
}

}  // namespace vfg

// ------------------------------------------------- persistent multi-problem apply
namespace vfg {


// Persistent walk over a work list.  dcount (optional) holds the item count on
// the device, so a captured graph follows a list that changes between replays;
// flags (optional) skip items of members whose flags[p * fstride] is 0.
// Schedules (the autotuner's choice): TX x TY element tiles of (TX-1) x (TY-1)
// owned node columns.  UNIT: the records are coarse multigrid levels.
template <typename T, int TX, int TY, bool UNIT, bool CUBIC>
__global__ __launch_bounds__(TX *TY, um_waves<T>()) void k_batch_u_apply(
    const BApply<T> *__restrict__ probs, const BItem *__restrict__ items, int nitems, const int *__restrict__ dcount,
    const double *__restrict__ flags, int fstride) {
  const int n = dcount ? *dcount : nitems;
  for (int it = blockIdx.x; it < n; it += gridDim.x) {
    const BItem w = items[it];
    if (flags && flags[(int64_t)w.p * fstride] == 0.) continue;  // uniform per block
    const auto op = op_of<UModOp<T, UNIT, CUBIC>>(probs[w.p].op);
    const int OZ = probs[w.p].OZ;
    __syncthreads();  // LDS of the previous item is free
    march_modal<TX, TY>(op.G, op, OZ, w.bx, w.by, w.bz);
  }
}

// schedule -> tile: 0: 16 x 16, 1: 8 x 8, 2: 16 x 8
int batch_tile_x(int sched) { return sched == 1 ? 8 : 16; }
int batch_tile_y(int sched) { return sched == 0 ? 16 : 8; }
template <typename T>
static int batch_slots_t(int sched) {
  if (sched == 1) return device_slots(k_batch_u_apply<T, 8, 8, false, false>, 64);
  if (sched == 2) return device_slots(k_batch_u_apply<T, 16, 8, false, false>, 128);
  return device_slots(k_batch_u_apply<T, 16, 16, false, false>, 256);
}
int batch_slots_s(int fp32, int sched) {
  static int cache[2][BATCH_SCHEDS] = {{0}};
  int &c = cache[fp32 ? 1 : 0][sched];
  if (!c) c = fp32 ? batch_slots_t<float>(sched) : batch_slots_t<double>(sched);
  return c;
}

size_t batch_op_bytes(int fp32) { return fp32 ? sizeof(BApply<float>) : sizeof(BApply<double>); }

int choose_oz_pub(const Grid &G, int tiles_xy, int slots) { return choose_oz(G, tiles_xy, slots); }

int batch_slots(int fp32) { return batch_slots_s(fp32, 0); }

template <typename T>
static void fill_ops_t(const std::vector<vfg_handle *> &m, const void *const *x, void *const *y,
                       const std::vector<int> &oz, void *d_ops, hipStream_t s) {
  std::vector<BApply<T>> ops(m.size());
  for (size_t p = 0; p < m.size(); p++) {
    const DevProblem &P = m[p]->P;
    umod_fill<T>(ops[p].op, P, (const T *)x[p], (T *)y[p]);
    ops[p].OZ = oz[p];
  }
  hipStreamSynchronize(s);  // no kernel of the previous call still reads d_ops
  hipMemcpy(d_ops, ops.data(), sizeof(BApply<T>) * ops.size(), hipMemcpyHostToDevice);
}

void fill_ops(const std::vector<vfg_handle *> &m, const void *const *x, void *const *y, int fp32,
              const std::vector<int> &oz, void *d_ops, hipStream_t s) {
  if (fp32) fill_ops_t<float>(m, x, y, oz, d_ops, s);
  else fill_ops_t<double>(m, x, y, oz, d_ops, s);
}

void launch_batch_apply(int fp32, int sched, int form, const void *d_ops, const BItem *items, int nitems, int grid,
                        hipStream_t s) {
  const int g = grid > 0 && grid < nitems ? grid : nitems;
  launch_engine_u_apply(fp32, sched, form, d_ops, items, nitems, nullptr, g, nullptr, 0, s);
}

template <typename T, int TX, int TY, bool UNIT>
static void launch_batch_t(bool cubic, const void *d_ops, const BItem *items, int nitems, const int *dcount, int grid,
                           const double *flags, int fstride, hipStream_t s) {
  auto go = [&](auto k) {
    hipLaunchKernelGGL(k, dim3(grid), dim3(TX * TY), 0, s, (const BApply<T> *)d_ops, items, nitems, dcount, flags,
                       fstride);
  };
  cubic ? go(k_batch_u_apply<T, TX, TY, UNIT, true>) : go(k_batch_u_apply<T, TX, TY, UNIT, false>);
}
template <typename T>
static void launch_batch_s(int sched, bool cubic, const void *d_ops, const BItem *items, int nitems, const int *dcount,
                           int grid, const double *flags, int fstride, hipStream_t s) {
  if (sched == 1) launch_batch_t<T, 8, 8, false>(cubic, d_ops, items, nitems, dcount, grid, flags, fstride, s);
  else if (sched == 2) launch_batch_t<T, 16, 8, false>(cubic, d_ops, items, nitems, dcount, grid, flags, fstride, s);
  else launch_batch_t<T, 16, 16, false>(cubic, d_ops, items, nitems, dcount, grid, flags, fstride, s);
}
void launch_engine_u_apply(int fp32, int sched, int form, const void *d_ops, const BItem *items, int nitems,
                           const int *dcount, int grid, const double *flags, int fstride, hipStream_t s) {
  const bool cubic = form & FORM_CUBIC;
  if (form & FORM_UNIT) launch_batch_t<float, 16, 16, true>(cubic, d_ops, items, nitems, dcount, grid, flags, fstride, s);
  else if (fp32) launch_batch_s<float>(sched, cubic, d_ops, items, nitems, dcount, grid, flags, fstride, s);
  else launch_batch_s<double>(sched, cubic, d_ops, items, nitems, dcount, grid, flags, fstride, s);
}

// multigrid smoothing records and their persistent launch
struct BSmooth {
  UMgRec op;
  int OZ;
};
template <class Op>
__global__ __launch_bounds__(256, 3) void k_batch_mg_smooth(const BSmooth *__restrict__ recs,
                                                            const BItem *__restrict__ items,
                                                            const int *__restrict__ dcount,
                                                            const double *__restrict__ flags, int fstride) {
  const int n = *dcount;
  for (int it = blockIdx.x; it < n; it += gridDim.x) {
    const BItem w = items[it];
    if (flags && flags[(int64_t)w.p * fstride] == 0.) continue;  // uniform per block
    const Op op = op_of<Op>(recs[w.p].op);
    const int OZ = recs[w.p].OZ;
    __syncthreads();  // LDS of the previous item is free
    march_modal<16, 16>(op.G, op, OZ, w.bx, w.by, w.bz);
  }
}
size_t mg_smooth_op_bytes() { return sizeof(BSmooth); }
void make_mg_smooth_op(const DevProblem &P, int post, const float *b, const float *dinv, float c2, const float *xin,
                       float *xo, float *ro, int OZ, void *out) {
  BSmooth r;
  mg_op_fill(r.op, P, b, dinv, c2);
  r.op.x = post ? xin : nullptr;
  r.op.xo = xo;
  r.op.ro = post ? nullptr : ro;
  r.OZ = OZ;
  *(BSmooth *)out = r;
}
void launch_batch_mg_smooth(int post, int form, const void *d_ops, const BItem *items, const int *dcount, int grid,
                            const double *flags, int fstride, hipStream_t s) {
  auto go = [&](auto k) {
    hipLaunchKernelGGL(k, dim3(grid), dim3(256), 0, s, (const BSmooth *)d_ops, items, dcount, flags, fstride);
  };
  const int f = form & (FORM_UNIT | FORM_CUBIC);
  if (post) {
    if (f == (FORM_UNIT | FORM_CUBIC)) go(k_batch_mg_smooth<UMgPostOp<true, false, true>>);
    else if (f == FORM_UNIT) go(k_batch_mg_smooth<UMgPostOp<true, false>>);
    else if (f == FORM_CUBIC) go(k_batch_mg_smooth<UMgPostOp<false, false, true>>);
    else go(k_batch_mg_smooth<UMgPostOp<false, false>>);
  } else {
    if (f == (FORM_UNIT | FORM_CUBIC)) go(k_batch_mg_smooth<UMgPreOp<true, true>>);
    else if (f == FORM_UNIT) go(k_batch_mg_smooth<UMgPreOp<true>>);
    else if (f == FORM_CUBIC) go(k_batch_mg_smooth<UMgPreOp<false, true>>);
    else go(k_batch_mg_smooth<UMgPreOp<false>>);
  }
}

// one member's operator entry for a persistent list (host memory `out`)
void make_uop(const DevProblem &P, const void *x, void *y, int fp32, int OZ, void *out) {
  if (fp32) {
    BApply<float> *b = (BApply<float> *)out;
    umod_fill<float>(b->op, P, (const float *)x, (float *)y);
    b->OZ = OZ;
  } else {
    BApply<double> *b = (BApply<double> *)out;
    umod_fill<double>(b->op, P, (const double *)x, (double *)y);
    b->OZ = OZ;
  }
}

}  // namespace vfg
