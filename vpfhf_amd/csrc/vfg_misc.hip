// vfg_misc.hip -- BC kit, energies / crack volume, penny cracks and the
// vector kernels of the solvers.  All reductions are two-stage with a fixed
// summation order, so results are bitwise reproducible run to run.
#include "vfg_modal.h"
#include "vfg_stage.h"
#include "vfg_kernels.h"

namespace vfg {

// ----------------------------------------------------------------- BC kit
struct BcTable {
  uint8_t face[3][6], vert[3][8];
  double faceValue[3][6], vertValue[3][8];
  int dof;
};
static BcTable bc_table(const DevProblem &P, int which) {
  BcTable t;
  t.dof = which == 0 ? 3 : 1;
  for (int c = 0; c < t.dof; c++) {
    const vfg_bc &b = which == 0 ? P.hbcU[c] : P.hbcV;
    for (int f = 0; f < 6; f++) { t.face[c][f] = (uint8_t)b.face[f]; t.faceValue[c][f] = b.faceValue[f]; }
    for (int v = 0; v < 8; v++) { t.vert[c][v] = (uint8_t)b.vertex[v]; t.vertValue[c][v] = b.vertex[v] ? b.vertexValue[v] : 0.; }
  }
  return t;
}

// Last writer over faces X0,X1,Y0,Y1,Z0,Z1 then the vertex (VFCartFE.c:279-483,
// 493-738).  Returns the BC type (0 if the dof is free) and the value it
// writes: FIXED takes faceValue/vertexValue (mode 0, VecSetFromBC) or B[d]
// (mode 1, VecApplyDirichletBC).
// With alias (vec and B are the same array, as in VecApplyDirichletBC(V,V,bcV)
// of VFTimeStepPrepare, VFCommon.c:1146) a FIXED entity copies the value the
// previous writer just stored, exactly as the in-place reference loops do.
__device__ int bc_last(const Grid &G, const BcTable &t, int c, int i, int j, int k, double Bd, int mode,
                       int alias, double *val) {
  int ty = 0;
  double v = Bd;
  const bool onf[6] = {i == 0, i == G.nx - 1, j == 0, j == G.ny - 1, k == 0, k == G.nz - 1};
  for (int f = 0; f < 6; f++)
    if (t.face[c][f] && onf[f]) {
      ty = t.face[c][f];
      v = ty == VFG_ZERO ? 0. : ty == VFG_ONE ? 1. : (mode == 0 ? t.faceValue[c][f] : alias ? v : Bd);
    }
  int ix = (i == 0) ? 0 : (i == G.nx - 1) ? 1 : -1;
  int iy = (j == 0) ? 0 : (j == G.ny - 1) ? 1 : -1;
  int iz = (k == 0) ? 0 : (k == G.nz - 1) ? 1 : -1;
  if (ix >= 0 && iy >= 0 && iz >= 0) {
    int vv = ix + 2 * iy + 4 * iz;
    if (t.vert[c][vv]) {
      ty = t.vert[c][vv];
      v = ty == VFG_ZERO ? 0. : ty == VFG_ONE ? 1. : (mode == 0 ? t.vertValue[c][vv] : alias ? v : Bd);
    }
  }
  *val = ty ? v : 0.;
  return ty;
}

__global__ void k_bc_vec(Grid G, BcTable t, uint8_t *mask, double *vec, const double *B, int mode) {
  const int alias = (mode == 1 && (const double *)vec == B);
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (int64_t)G.nx * G.ny * G.nz) return;
  int i = (int)(n % G.nx), j = (int)((n / G.nx) % G.ny), k = (int)(n / ((int64_t)G.nx * G.ny));
  for (int c = 0; c < t.dof; c++) {
    int64_t d = t.dof * n + c;
    double val;
    int ty = bc_last(G, t, c, i, j, k, B ? B[d] : 0., mode, alias, &val);
    if (mask) mask[d] = ty ? 1 : 0;
    if (vec && ty) vec[d] = val;
  }
}

static unsigned nblk(int64_t n, int bs = 256) { return (unsigned)((n + bs - 1) / bs); }

void launch_bc_mask(const DevProblem &P, int which, uint8_t *mask, hipStream_t s) {
  hipLaunchKernelGGL(k_bc_vec, dim3(nblk(P.nn)), dim3(256), 0, s, P.G, bc_table(P, which), mask,
                     (double *)nullptr, (const double *)nullptr, 0);
}
void launch_vec_set_from_bc(const DevProblem &P, int which, double *B, hipStream_t s) {
  hipLaunchKernelGGL(k_bc_vec, dim3(nblk(P.nn)), dim3(256), 0, s, P.G, bc_table(P, which),
                     (uint8_t *)nullptr, B, (const double *)nullptr, 0);
}
void launch_vec_apply_dirichlet(const DevProblem &P, int which, double *vec, const double *B, hipStream_t s) {
  hipLaunchKernelGGL(k_bc_vec, dim3(nblk(P.nn)), dim3(256), 0, s, P.G, bc_table(P, which),
                     (uint8_t *)nullptr, vec, B, 1);
}

// ------------------------------------------------------- energies / volume
// Per element (VFMech.c:725-809, 920-974, 2394-2465; VFPermfield.c:15-71):
//   elastic = sum_g W [mu(1+eta) v^2 |e^D|^2 + 3(3lam+2mu)/2 ((tr/3 - alpha dth) v
//             - beta p/(3lam+2mu))^2 + (3lam+2mu)/6 tr^2 eta]
//   pressure work = sum_g W p (u . grad v)
//   surface = Gc/(4 atCv) sum_g W [(1-v)^k/eps + eps |grad v|^2], k = 1 (AT1), 2 (AT2)
//   crack volume = sum_g W u . grad v
// A workgroup takes a 16 x 16 tile of element columns over EZ element layers
// (energy_layers):
// the node planes (u, v, p, theta - thetaRef) are staged in LDS two at a time,
// the next one loaded into registers meanwhile, and each thread evaluates its
// element from the modal sums of its corners (vfg_modal.h).  One group of 4
// partials per workgroup, in a fixed order.
constexpr int EB = 256, ET = 16, EP = ET + 1;
// the operators' constants, formed once on the host (kernel arguments sit in
// scalar registers; formed in the kernel they take vector ones)
struct EnergyConst {
  double kx, ky;        // d_x, d_y relative to d_z
  double kt[3];         // a third of the derivative per modal sum
  double kc[3], kp[3];  // opening and pressure work
  double ks[8];         // surface energy per squared modal sum of v; [0]: of the mean of 1 - v or its square
  double dev, sph, tr2, cb, ivol;
};
static EnergyConst energy_const(const DevProblem &P) {
  const Grid &G = P.G;
  const double vol = G.hx * G.hy * G.hz, ih[3] = {1. / G.hx, 1. / G.hy, 1. / G.hz}, tk1 = 3. * P.lam1 + 2. * P.mu1;
  const double csurf = P.Gc / P.atcv * .25 * vol;
  EnergyConst C;
  for (int d = 0; d < 3; d++) {
    C.kt[d] = ih[d] / 12.;
    C.kc[d] = ih[d] * vol / 32.;
    C.kp[d] = ih[d] * vol / 256.;
  }
  C.kx = G.hz / G.hx;
  C.ky = G.hz / G.hy;
  C.ks[0] = csurf / P.eps;
  for (int i = 1; i < 8; i++) {
    const int o = __builtin_popcount(i);
    double kk = 0.;
    for (int d = 0; d < 3; d++)
      if (um_pow(i, d)) kk += ih[d] * ih[d] / (o == 1 ? 1. : o == 2 ? 3. : 9.);
    C.ks[i] = csurf * P.eps / 16. * kk + (P.atnum == 2 ? C.ks[0] / (64. * (o == 1 ? 3. : o == 2 ? 9. : 27.)) : 0.);
  }
  C.dev = vol * P.mu1 * (1. + P.eta) / 64. * (ih[2] * ih[2] / 16.);
  C.sph = vol * 1.5 * tk1 / 64.;
  C.tr2 = vol * 1.5 * tk1 * P.eta;
  C.cb = P.beta / tk1;
  C.ivol = 1. / vol;
  return C;
}

// sum_g W u . grad v of an element from the modal sums of u and v
__device__ __forceinline__ double opening_work(const double (&U)[3][8], const double (&V)[8],
                                               const EnergyConst &C) {
  double s = 0.;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    double t = 0.;
#pragma unroll
    for (int q = 3; q >= 0; q--) {  // <u_d d_d v>: the other variables' squares average 1/3 each
      const int b = q & 1, c = q >> 1;
      t += (b + c == 2 ? 1. / 9. : b + c ? 1. / 3. : 1.) * (U[d][modal_at(d, 0, b, c)] * V[modal_at(d, 1, b, c)]);
    }
    s += C.kc[d] * t;
  }
  return s;
}
// sum_g W p (u . grad v): along d the average of p u_d, times d_d v, over the
// Gauss points of the two other variables
__device__ __forceinline__ double pressure_work(const double (&U)[3][8], const double (&V)[8], const double (&Pm)[8],
                                                const EnergyConst &C) {
  double s = 0.;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    double t = 0.;
#pragma unroll
    for (int g2 = 0; g2 < 3; g2++) {
      double p[2][2], u[2][2], v[2];  // [power of variable d][power of the second variable]
#pragma unroll
      for (int b = 0; b < 2; b++) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
          p[q][b] = at_gauss(g2, Pm[modal_at(d, q, b, 0)], Pm[modal_at(d, q, b, 1)]);
          u[q][b] = at_gauss(g2, U[d][modal_at(d, q, b, 0)], U[d][modal_at(d, q, b, 1)]);
        }
        v[b] = at_gauss(g2, V[modal_at(d, 1, b, 0)], V[modal_at(d, 1, b, 1)]);
      }
#pragma unroll
      for (int g1 = 0; g1 < 3; g1++) {
        const double pu = at_gauss(g1, p[0][0], p[0][1]) * at_gauss(g1, u[0][0], u[0][1]) +
                          (1. / 3.) * (at_gauss(g1, p[1][0], p[1][1]) * at_gauss(g1, u[1][0], u[1][1]));
        t += gW(g1) * gW(g2) * (pu * at_gauss(g1, v[0], v[1]));
      }
    }
    s += C.kp[d] * t;
  }
  return s;
}
// sum_g w v^2 |e^D|^2 from the modal sums, times 64 (4 hz)^2
__device__ __forceinline__ double deviatoric(const double (&U)[3][8], const double (&V)[8],
                                             const EnergyConst &C) {
  double s = 0.;
#pragma unroll 1
  for (int gz = 0; gz < 3; gz++) {  // a loop of its own per layer of points: registers
    const double x = gz == 0 ? gX(0) : gz == 1 ? 0. : gX(2);
    double dx[3][2], dy[3][3], v[4];  // strains in units of d_z's factor: that derivative takes U as it is
#pragma unroll
    for (int c = 0; c < 3; c++) {
#pragma unroll
      for (int b = 0; b < 2; b++) dx[c][b] = C.kx * (U[c][1 + 2 * b] + x * U[c][5 + 2 * b]);
      const double y0 = C.ky * (U[c][2] + x * U[c][6]), y1 = C.ky * (U[c][3] + x * U[c][7]);
#pragma unroll
      for (int gx = 0; gx < 3; gx++) dy[c][gx] = at_gauss(gx, y0, y1);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = (V[q] + x * V[q + 4]);
#pragma unroll
    for (int gy = 0; gy < 3; gy++) {
      double hx[3], z0[3], z1[3], row = 0.;
#pragma unroll
      for (int c = 0; c < 3; c++) {
        hx[c] = at_gauss(gy, dx[c][0], dx[c][1]);
        z0[c] = at_gauss(gy, U[c][4], U[c][6]);
        z1[c] = at_gauss(gy, U[c][5], U[c][7]);
      }
      const double v0 = at_gauss(gy, v[0], v[2]), v1 = at_gauss(gy, v[1], v[3]);
#pragma unroll
      for (int gx = 0; gx < 3; gx++) {
        const double vg = at_gauss(gx, v0, v1), e22 = dy[1][gx], e33 = at_gauss(gx, z0[2], z1[2]);
        const double t01 = dy[0][gx] + hx[1], t02 = at_gauss(gx, z0[0], z1[0]) + hx[2],
                     t12 = at_gauss(gx, z0[1], z1[1]) + dy[2][gx];
        // the diagonal of e^D through its differences: 2/3 (a^2 + a b + b^2)
        const double a = hx[0] - e22, b = e22 - e33;
        const double dev = (2. / 3.) * (a * (a + b) + b * b) + .5 * (t01 * t01 + t02 * t02 + t12 * t12);
        row += gW(gx) * (vg * vg) * dev;
      }
      s += gW(gy) * (gz == 1 ? gW(1) : gW(0)) * row;
    }
  }
  return s;
}
// sum_g w (tr/3 v - alpha dth v - q)^2, tr/3 by its modal sums R (no xyz term),
// T = 8 alpha dth, Q = 8 q; times 64.  UNILATERAL_NOCOMPRESSION: v = 1 where
// tr(eps) < 0 (VF_ElasticEnergyNoCompression3D_local, VFMech.c:871-903)
template <bool UNI>
__device__ __forceinline__ double spherical(const double (&R)[7], const double (&V)[8], const double (&T)[8],
                                            const double (&Q)[8]) {
  double s = 0.;
#pragma unroll
  for (int gz = 0; gz < 3; gz++) {
    double f[4][4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      f[0][q] = at_gauss(gz, V[q], V[q + 4]);
      f[1][q] = at_gauss(gz, T[q], T[q + 4]);
      f[2][q] = at_gauss(gz, Q[q], Q[q + 4]);
      f[3][q] = q == 3 ? R[3] : at_gauss(gz, R[q], R[q + 4]);
    }
#pragma unroll
    for (int gy = 0; gy < 3; gy++) {
      double r[4][2], row = 0.;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        r[c][0] = at_gauss(gy, f[c][0], f[c][2]);
        r[c][1] = at_gauss(gy, f[c][1], f[c][3]);
      }
#pragma unroll
      for (int gx = 0; gx < 3; gx++) {
        double p[4];
#pragma unroll
        for (int c = 0; c < 4; c++) p[c] = at_gauss(gx, r[c][0], r[c][1]);
        const double v = UNI && p[3] < 0. ? 8. : p[0], w = (p[3] - .125 * p[1]) * v - p[2];
        row += gW(gx) * (w * w);
      }
      s += gW(gy) * gW(gz) * row;
    }
  }
  return s;
}

// Bound by FP64 issue at two waves per SIMD: about 1350 operations per element
// against 2900 when every field and gradient is interpolated from the corners
// at each of the 27 points.  113 x 126 x 98: 99 us, 300 us so (eight layers).
// Registers decide here: at three waves per SIMD 86 of them spill (254 us).
template <bool UNI>
__global__ __launch_bounds__(EB, 2) void k_energies(DevProblem P, EnergyConst C, const double *__restrict__ U,
                                                    const double *__restrict__ V, double *partials,
                                                    double *cellfield, double *efield, int EZ) {
  __shared__ double sp[3][6][EP * EP];  // three planes: one barrier per layer
  __shared__ double sh[EB / 64];
  const Grid &G = P.G;
  const int tid = threadIdx.x, tx = tid % ET, ty = tid / ET;
  const Blk3 bk = xcd_block();
  const int ex0 = bk.x * ET, ey0 = bk.y * ET, ek0 = bk.z * EZ;
  const int ek1 = min(ek0 + EZ, G.nez);
  const int ex = ex0 + tx, ey = ey0 + ty;
  const bool ok = ex < G.nex && ey < G.ney;
  // fields 0-2: u_c, 3: v, 4: p, 5: theta - thetaRef
  // each thread takes one node of the tile's first 16 x 16, and one value of the rest
  const bool in = ex < G.nx && ey < G.ny;
  const int hf = tid / (EP * EP - EB), hq = tid % (EP * EP - EB);  // field; node of the last column, then row
  const int hi = hq < EP ? ET : hq - EP, hj = hq < EP ? hq : ET;
  const bool hin = hf < 6 && ex0 + hi < G.nx && ey0 + hj < G.ny;
  const double *const hp = hf < 3 ? U + hf : hf == 3 ? V : hf == 4 ? P.p : P.dth;
  double pf[6] = {0., 0., 0., 0., 0., 0.}, ph = 0.;
  auto fetch = [&](int k) {
    if (in) {
      const int64_t n = node_id(G, ex, ey, k);
#pragma unroll
      for (int c = 0; c < 3; c++) pf[c] = U[3 * n + c];
      pf[3] = V[n];
      pf[4] = P.p[n];
      pf[5] = P.dth[n];
    }
    if (hin) ph = hp[node_id(G, ex0 + hi, ey0 + hj, k) * (hf < 3 ? 3 : 1)];
  };
  auto commit = [&](int b) {
#pragma unroll
    for (int f = 0; f < 6; f++) sp[b][f][ty * EP + tx] = pf[f];
    if (hf < 6) sp[b][hf][hj * EP + hi] = ph;
  };
  double el = 0., pw = 0., se = 0., cv = 0.;
  fetch(ek0);
  commit(0);
  fetch(ek0 + 1);
  for (int ek = ek0; ek < ek1; ek++) {
    const int b = (ek - ek0) % 3, b1 = (ek + 1 - ek0) % 3;
    commit(b1);  // plane ek + 1, over ek - 2, last read before the barrier of layer ek - 1
    if (ek + 1 < ek1) fetch(ek + 2);
    __syncthreads();
    if (ok) {
      const int64_t e = cell_id(G, ex, ey, ek);
      const double Ee = P.E_elem ? P.E_elem[e] : P.E;
      const int c0 = ty * EP + tx;
      auto sums = [&](int q, double (&m)[8]) {
        modal_sums([&](int a) { return sp[(a >> 2) ? b1 : b][q][c0 + ((a >> 1) & 1) * EP + (a & 1)]; }, m);
      };
      double Vm[8], R[7], cell, cel, cpw = 0., cse, tr2 = 0.;
      sums(3, Vm);
      {
        double Um[3][8];
#pragma unroll
        for (int c = 0; c < 3; c++) sums(c, Um[c]);
        cell = opening_work(Um, Vm, C);
        if (P.hasCrackPressure) {
          double Pm[8];
          sums(4, Pm);
          cpw = pressure_work(Um, Vm, Pm, C);
        }
        asm volatile("" ::: "memory");  // p is read again below rather than held: registers
        // modal sums of tr/3; no two of them share a point average
#pragma unroll
        for (int i = 0; i < 7; i++) {
          double t = 0.;
#pragma unroll
          for (int d = 0; d < 3; d++)
            if (!um_pow(i, d)) t += C.kt[d] * Um[d][i | 1 << d];
          R[i] = t;
          const int o = __builtin_popcount(i);
          tr2 += (o == 2 ? 1. / 9. : o ? 1. / 3. : 1.) * (t * t);
        }
        __builtin_amdgcn_sched_barrier(0);
        cel = C.dev * deviatoric(Um, Vm, C);
      }
      {  // 1 - v (AT1) or its square (AT2), and |grad v|^2: orthogonal in the modal sums
        const double om = 1. - .125 * Vm[0];
        cse = C.ks[0] * (P.atnum == 2 ? om * om : om);
#pragma unroll
        for (int i = 1; i < 8; i++) cse += C.ks[i] * (Vm[i] * Vm[i]);
      }
      {  // 3 tk/2 ((tr/3 - alpha dth) v - beta p/tk)^2 + tk/6 tr^2 eta, tk = 3 lam + 2 mu
        double Tm[8], Qm[8];
        sums(5, Tm);
        sums(4, Qm);
        const double cb = C.cb / Ee;
#pragma unroll
        for (int q = 0; q < 8; q++) {
          Tm[q] *= P.alpha;
          Qm[q] *= cb;
        }
        cel += C.sph * spherical<UNI>(R, Vm, Tm, Qm) + C.tr2 * tr2;
        cel *= Ee;
      }
      el += cel; pw += cpw; se += cse; cv += cell;
      if (cellfield) cellfield[e] = cell * C.ivol;
      if (efield) {
        efield[3 * e] = cel;
        efield[3 * e + 1] = cpw;
        efield[3 * e + 2] = cse;
      }
    }
  }
  double r0 = block_sum<EB>(el, sh), r1 = block_sum<EB>(pw, sh), r2 = block_sum<EB>(se, sh),
         r3 = block_sum<EB>(cv, sh);
  if (tid == 0) {
    const int64_t blk = bk.x + (int64_t)gridDim.x * (bk.y + (int64_t)gridDim.y * bk.z);  // partials in block order
    partials[blk * 4 + 0] = r0; partials[blk * 4 + 1] = r1;
    partials[blk * 4 + 2] = r2; partials[blk * 4 + 3] = r3;
  }
}

// The crack volume and the opening per cell alone: u and v of the element's
// corners straight from memory (each line is reused from the caches by the
// neighbouring lanes and rows), the upper plane's values kept for the next
// layer.  Bound by the read of u and v: 113 x 126 x 98 in 19 us, against the
// whole of k_energies.
__global__ __launch_bounds__(EB) void k_crack_volume(Grid G, EnergyConst C, const double *__restrict__ U, const double *__restrict__ V,
                                                     double *__restrict__ partials, double *__restrict__ cellfield,
                                                     int EZ) {
  __shared__ double sh[EB / 64];
  const int tx = threadIdx.x % ET, ty = threadIdx.x / ET;
  const Blk3 bk = xcd_block();
  const int ex = bk.x * ET + tx, ey = bk.y * ET + ty, ek0 = bk.z * EZ, ek1 = min(ek0 + EZ, G.nez);
  double cv = 0.;
  if (ex < G.nex && ey < G.ney) {
    double f[4][8];
    auto plane = [&](int k, int o) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int64_t n = node_id(G, ex + (q & 1), ey + (q >> 1), k);
#pragma unroll
        for (int c = 0; c < 3; c++) f[c][o + q] = U[3 * n + c];
        f[3][o + q] = V[n];
      }
    };
    plane(ek0, 0);
    for (int ek = ek0; ek < ek1; ek++) {
      plane(ek + 1, 4);
      double Um[3][8], Vm[8];
#pragma unroll
      for (int c = 0; c < 3; c++) modal_sums([&](int a) { return f[c][a]; }, Um[c]);
      modal_sums([&](int a) { return f[3][a]; }, Vm);
      const double cell = opening_work(Um, Vm, C);
      cv += cell;
      if (cellfield) cellfield[cell_id(G, ex, ey, ek)] = cell * C.ivol;
#pragma unroll
      for (int c = 0; c < 4; c++)
#pragma unroll
        for (int q = 0; q < 4; q++) f[c][q] = f[c][q + 4];
    }
  }
  const double r = block_sum<EB>(cv, sh);
  if (threadIdx.x == 0) partials[bk.x + (int64_t)gridDim.x * (bk.y + (int64_t)gridDim.y * bk.z)] = r;
}

// sums `nb` groups of W partials column-wise with one block
template <int W>
__global__ __launch_bounds__(256) void k_reduce_partials(const double *__restrict__ partials, int nb,
                                                         double *__restrict__ out) {
  __shared__ double sh[4];
  double s[W] = {};
  for (int b = threadIdx.x; b < nb; b += 256)
#pragma unroll
    for (int c = 0; c < W; c++) s[c] += partials[(int64_t)b * W + c];
#pragma unroll
  for (int c = 0; c < W; c++) {
    const double r = block_sum<256>(s[c], sh);
    if (threadIdx.x == 0) out[c] = r;
  }
}

int device_slots_of(const void *kernel, int threads);  // vfg_u.hip
static int64_t element_tiles(const Grid &G) { return (int64_t)((G.nex + ET - 1) / ET) * ((G.ney + ET - 1) / ET); }
static dim3 layer_grid(const Grid &G, int ez) {
  return dim3((G.nex + ET - 1) / ET, (G.ney + ET - 1) / ET, (G.nez + ez - 1) / ez);
}
// layers per workgroup of the crack volume, which is bound by memory
static int volume_layers(const Grid &G) { return element_tiles(G) >= 64 ? 8 : 2; }
// of the energies: the fewest whole rounds of resident workgroups times layers
// (and one for the first plane and the sums), as for the marches.  Eight layers
// whatever the grid left a second round of 113 x 126 x 98 elements half empty:
// 115 us against 99 (thirteen layers; 3 to 14 layers 95 to 120).
// Chunks under eight layers only while their partials fit a handle's own array.
static int energy_layers(const DevProblem &P) {
  static const int slots_uni = device_slots_of((const void *)k_energies<true>, EB);
  static const int slots_lin = device_slots_of((const void *)k_energies<false>, EB);
  const int slots = P.unilateral ? slots_uni : slots_lin;
  const int64_t tiles = element_tiles(P.G);
  int best = 8;
  int64_t best_cost = INT64_MAX;
  for (int ez = 1; ez <= P.G.nez; ez++) {
    const int chunks = (P.G.nez + ez - 1) / ez;
    if (ez > 1 && (P.G.nez + ez - 2) / (ez - 1) == chunks) continue;  // same chunk count, shorter is free
    if (ez < 8 && tiles * chunks > 65536) continue;
    const int64_t cost = (tiles * chunks + slots - 1) / slots * (ez + 1);
    if (cost < best_cost) best_cost = cost, best = ez;
  }
  return best;
}
int64_t energy_cell_blocks(const DevProblem &P) {
  const dim3 g = layer_grid(P.G, volume_layers(P.G));
  return (int64_t)g.x * g.y * g.z;
}
int energy_blocks(const DevProblem &P) {
  const dim3 g = layer_grid(P.G, energy_layers(P));
  return (int)std::max((int64_t)g.x * g.y * g.z, energy_cell_blocks(P));
}

void launch_energies(const DevProblem &P, const double *U, const double *V, double *partials,
                     double *cellfield, double *efield, double *result4, hipStream_t s) {
  const int ez = energy_layers(P);
  const dim3 g = layer_grid(P.G, ez);
  auto go = [&](auto k) {
    hipLaunchKernelGGL(k, g, dim3(EB), 0, s, P, energy_const(P), U, V, partials, cellfield, efield, ez);
  };
  P.unilateral ? go(k_energies<true>) : go(k_energies<false>);
  hipLaunchKernelGGL(k_reduce_partials<4>, dim3(1), dim3(256), 0, s, (const double *)partials, (int)(g.x * g.y * g.z),
                     result4);
}
void launch_crack_volume(const DevProblem &P, const double *U, const double *V, double *partials, double *cellfield,
                         double *result, hipStream_t s) {
  const int ez = volume_layers(P.G);
  const dim3 g = layer_grid(P.G, ez);
  hipLaunchKernelGGL(k_crack_volume, g, dim3(EB), 0, s, P.G, energy_const(P), U, V, partials, cellfield, ez);
  hipLaunchKernelGGL(k_reduce_partials<1>, dim3(1), dim3(256), 0, s, (const double *)partials, (int)(g.x * g.y * g.z),
                     result);
}

// ------------------------------------------------------------ staged uploads
// one segment per blockIdx.x
__global__ __launch_bounds__(256) void k_stage(const StageSeg *__restrict__ seg) {
  const StageSeg q = seg[blockIdx.x];
  const size_t n = q.bytes / 4, st = (size_t)gridDim.y * 256;
  uint32_t *__restrict__ d = (uint32_t *)q.dst;
  const uint32_t *__restrict__ a = (const uint32_t *)q.src;
  for (size_t i = (size_t)blockIdx.y * 256 + threadIdx.x; i < n; i += st) d[i] = a[i];
}
void launch_stage(const StageSeg *seg, int n, size_t max_bytes, hipStream_t s) {
  const unsigned ny = (unsigned)((max_bytes + 4095) / 4096);
  hipLaunchKernelGGL(k_stage, dim3(n, ny < 1 ? 1 : ny > 64 ? 64 : ny), dim3(256), 0, s, seg);
}

// ------------------------------------------------------------ penny crack
// VFDistanceToPennyCrack + VFPennyCrackBuildVAT1/AT2 (VFCracks.c:101-227);
// node coordinates X[i] = i*lx/(nx-1) (VFCommon.c:395-397).
__global__ void k_penny(Grid G, double lx, double ly, double lz, int atnum, double eps, double *V,
                        double c0, double c1, double c2, double r, double th, double ph, double thick) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (int64_t)G.nx * G.ny * G.nz) return;
  int i = (int)(n % G.nx), j = (int)((n / G.nx) % G.ny), k = (int)(n / ((int64_t)G.nx * G.ny));
  double x0 = i == 0 ? 0. : i * lx / (G.nx - 1.);
  double x1 = j == 0 ? 0. : j * ly / (G.ny - 1.);
  double x2 = k == 0 ? 0. : k * lz / (G.nz - 1.);
  if (r == 0) { V[n] = 1.; return; }
  const double PI = 3.14159265358979323846;
  double nv0 = cos(th * PI / 180.) * sin(ph * PI / 180.);
  double nv1 = sin(th * PI / 180.) * sin(ph * PI / 180.);
  double nv2 = cos(ph * PI / 180.);
  double xdn = (x0 - c0) * nv0 + (x1 - c1) * nv1 + (x2 - c2) * nv2;
  double t0 = (x0 - c0) - xdn * nv0, t1 = (x1 - c1) - xdn * nv1, t2 = (x2 - c2) - xdn * nv2;
  double l = sqrt(t0 * t0 + t1 * t1 + t2 * t2);
  double dist = (l <= r) ? sqrt(xdn * xdn) : sqrt(xdn * xdn + (l - r) * (l - r));
  dist -= thick / 2.;
  double val;
  if (atnum == 1) val = dist <= 0 ? 0. : dist < 2. * eps ? dist / eps * (1. - .25 * dist / eps) : 1.;
  else val = dist <= 0 ? 0. : 1. - exp(-dist / 2 / eps);
  V[n] = val;
}

void launch_penny(const DevProblem &P, double *V, const double c[3], double r, double theta, double phi,
                  double thick, hipStream_t s) {
  double lx = P.G.hx * P.G.nex, ly = P.G.hy * P.G.ney, lz = P.G.hz * P.G.nez;
  hipLaunchKernelGGL(k_penny, dim3(nblk(P.nn)), dim3(256), 0, s, P.G, lx, ly, lz, P.atnum, P.eps, V,
                     c[0], c[1], c[2], r, theta, phi, thick);
}

// ------------------------------------------------- cell -> node averaging
// CellToNodeInterpolation (VFPermfield.c:1156-1327): every node takes the
// volume-weighted mean of its adjacent cells, node = sum(cell*hx*hy*hz) /
// sum(hz*hy*hx).  The reference scatters cell by cell; here each thread
// gathers one (node, component) pair, visiting the adjacent cells in the
// order the scatter reaches the node (ek, ej, ei ascending) with the same
// products and no contraction, so the sums round as the reference's do.
// Cell sizes come from the node coordinates X[i] = i*l/(n-1)
// (VFCommon.c:395-397), as the reference reads them from ctx->coordinates.
__device__ __forceinline__ double coord_of(int i, double l, int n) { return i == 0 ? 0. : i * l / (n - 1.); }

__global__ __launch_bounds__(256) void k_cell_to_node(Grid G, double lx, double ly, double lz, const double *cell,
                                                      double *node, int dof) {
#pragma clang fp contract(off)
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nn = (int64_t)G.nx * G.ny * G.nz;
  if (t >= nn * dof) return;
  const int64_t n = t / dof;
  const int d = (int)(t - n * dof);
  const int i = (int)(n % G.nx), j = (int)((n / G.nx) % G.ny), k = (int)(n / ((int64_t)G.nx * G.ny));
  double acc = 0., vol = 0.;
  for (int ek = k > 0 ? k - 1 : 0; ek <= k && ek < G.nez; ek++) {
    const double hz = coord_of(ek + 1, lz, G.nz) - coord_of(ek, lz, G.nz);
    for (int ej = j > 0 ? j - 1 : 0; ej <= j && ej < G.ney; ej++) {
      const double hy = coord_of(ej + 1, ly, G.ny) - coord_of(ej, ly, G.ny);
      for (int ei = i > 0 ? i - 1 : 0; ei <= i && ei < G.nex; ei++) {
        const double hx = coord_of(ei + 1, lx, G.nx) - coord_of(ei, lx, G.nx);
        vol = vol + hz * hy * hx;
        acc = acc + cell[dof * cell_id(G, ei, ej, ek) + d] * hx * hy * hz;
      }
    }
  }
  node[t] = acc / vol;
}

void launch_cell_to_node(const DevProblem &P, double lx, double ly, double lz, const double *cell, double *node,
                         int dof, hipStream_t s) {
  const int64_t n = P.nn * dof;
  hipLaunchKernelGGL(k_cell_to_node, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, P.G, lx, ly, lz, cell,
                     node, dof);
}

// ------------------------------------------------------------ vector ops
constexpr int RB = 256;
int red_blocks(int64_t n) {
  int64_t b = (n + RB * 4 - 1) / (RB * 4);
  return (int)(b < 1 ? 1 : b > 2048 ? 2048 : b);
}

__global__ __launch_bounds__(RB) void k_dot(const double *__restrict__ a, const double *__restrict__ b,
                                            int64_t n, double *partials) {
  __shared__ double sh[RB / 64];
  double s = 0.;
  for (int64_t i = (int64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB) s += a[i] * b[i];
  s = block_sum<RB>(s, sh);
  if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

void launch_dot(const double *a, const double *b, int64_t n, double *partials, double *out, hipStream_t s) {
  int nb = red_blocks(n);
  hipLaunchKernelGGL(k_dot, dim3(nb), dim3(RB), 0, s, a, b, n, partials);
  hipLaunchKernelGGL(k_reduce_partials<1>, dim3(1), dim3(256), 0, s, (const double *)partials, nb, out);
}

__global__ void k_fill(double *x, double v, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = v;
}
void launch_fill(double *x, double v, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_fill, dim3(nblk(n)), dim3(256), 0, s, x, v, n);
}
__global__ void k_sub(const double *a, const double *b, double *o, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) o[i] = a[i] - b[i];
}
void launch_sub(const double *a, const double *b, double *out, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_sub, dim3(nblk(n)), dim3(256), 0, s, a, b, out, n);
}
__global__ void k_d2f(const double *x, float *y, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = (float)x[i];
}
__global__ void k_f2d(const float *x, double *y, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = (double)x[i];
}
void launch_copy_d2f(const double *x, float *y, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_d2f, dim3(nblk(n)), dim3(256), 0, s, x, y, n);
}
void launch_copy_f2d(const float *x, double *y, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_f2d, dim3(nblk(n)), dim3(256), 0, s, x, y, n);
}

__global__ void k_vmin(const double *a, const double *b, double *o, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) o[i] = fmin(a[i], b[i]);
}
__global__ void k_scale(double *x, double s, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] *= s;
}
__global__ __launch_bounds__(RB) void k_maxabs(const double *a, const double *b, int64_t n, double *part) {
  __shared__ double sh[RB];
  double m = 0.;
  for (int64_t i = (int64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB)
    m = fmax(m, fabs(a[i] - b[i]));
  sh[threadIdx.x] = m;
  __syncthreads();
  for (int o = RB / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + o]);
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}
// max over the partials: one workgroup, strided loads, then a tree in LDS
// (max is exact, so any order gives the same value)
__global__ __launch_bounds__(RB) void k_maxreduce(const double *part, int nb, double *out) {
  __shared__ double sh[RB];
  double m = 0.;
  for (int i = threadIdx.x; i < nb; i += RB) m = fmax(m, part[i]);
  sh[threadIdx.x] = m;
  __syncthreads();
  for (int w = RB / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = sh[0];
}
void launch_vmin(const double *a, const double *b, double *o, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_vmin, dim3(nblk(n)), dim3(256), 0, s, a, b, o, n);
}
void launch_scale(double *x, double v, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_scale, dim3(nblk(n)), dim3(256), 0, s, x, v, n);
}
void launch_maxabs_diff(const double *a, const double *b, int64_t n, double *part, double *out, hipStream_t s) {
  int nb = red_blocks(n);
  hipLaunchKernelGGL(k_maxabs, dim3(nb), dim3(RB), 0, s, a, b, n, part);
  hipLaunchKernelGGL(k_maxreduce, dim3(1), dim3(RB), 0, s, (const double *)part, nb, out);
}

}  // namespace vfg

// ------------------------------------------- energies without allocation
// vfg_energies_static: the reductions of vfg_energies with their partials in
// a file-scope device array instead of handle buffers, for callers that
// cannot allocate device memory (HIP graph capture, serving loops, harnesses
// that forbid hipMalloc).  The array holds ENERGY_STATIC_BLOCKS groups of 4
// partials plus the 4 results: 8 MiB + 32 B, resident on every GPU the
// library runs on until the process ends.  Every partial is written by
// k_energies before k_reduce_partials reads it, so nothing needs clearing;
// calls that overlap on one GPU share the array and race.
#include <mutex>
#include "vfg_handle.h"

static constexpr int ENERGY_STATIC_BLOCKS = 1 << 18;  // workgroups of 16 x 16 x 8 cells: 536,870,912 cells
static __device__ __align__(256) double scratch[4 * ENERGY_STATIC_BLOCKS + 4];

namespace {
constexpr int MAX_DEVICES = 64;
// device address of `scratch` on each GPU (the host-side name is a stand-in,
// never a device address)
double *g_scratch_dev[MAX_DEVICES];
std::mutex g_scratch_mu;

int scratch_address(vfg_handle *h, double **out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES)
    return vfg_fail(h, VFG_E_HIP, "vfg_energies_static: no current HIP device (or device id >= %d)", MAX_DEVICES);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    void *p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return vfg_fail(h, VFG_E_HIP, "vfg_energies_static: hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    g_scratch_dev[dev] = (double *)p;
  }
  *out = g_scratch_dev[dev];
  return VFG_OK;
}
}  // namespace

extern "C" int vfg_energies_static(vfg_handle *h, const double *U, const double *V, double out[4]) {
  if (!h) return vfg_fail(nullptr, VFG_E_ARG, "NULL handle");
  if (!U || !V || !out) return vfg_fail(h, VFG_E_ARG, "vfg_energies_static: NULL array");
  // (the groups that are written are no more than these, or than 65536)
  const int64_t nb = vfg::energy_cell_blocks(h->P);
  if (nb > ENERGY_STATIC_BLOCKS)
    return vfg_fail(h, VFG_E_ARG,
                    "vfg_energies_static: %lld cells need %lld partial groups, more than the %d of the "
                    "static scratch array (use vfg_energies)",
                    (long long)h->P.ne, (long long)nb, ENERGY_STATIC_BLOCKS);
  double *part = nullptr;
  int rc = scratch_address(h, &part);
  if (rc) return rc;
  double *res = part + 4 * (size_t)ENERGY_STATIC_BLOCKS;
  vfg::launch_energies(h->P, U, V, part, nullptr, nullptr, res, h->stream);
  double r[4];
  if (hipMemcpyAsync(r, res, sizeof r, hipMemcpyDeviceToHost, h->stream) != hipSuccess ||
      hipStreamSynchronize(h->stream) != hipSuccess || hipGetLastError() != hipSuccess)
    return vfg_fail(h, VFG_E_HIP, "vfg_energies_static: kernel execution failed");
  out[0] = r[0];
  out[1] = 0.;
  out[2] = r[1];
  out[3] = r[2];
  return VFG_OK;
}
