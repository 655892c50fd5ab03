// vfg_v.hip -- V-subproblem (AT1/AT2 phase field) operators on gfx950.
//
// Element matrix (VFMech.c:2040-2115):
//   K[a][b] = c sum_g W_g (phi_a phi_b / eps [AT2 only] + eps grad phi_a . grad phi_b)
//           + sum_g W_g phi_a phi_b 2 W^el_g,            c = Gc / atCv / 2,
//   W^el_g = 1/2 sigma(e~):e~,  e~ = e(u) - alpha dtheta I  (VFMech.c:32-106).
// Split as K = ks * L + M_q with the Q1 stiffness L and the point-weighted mass
// M_q, q_g = W_g (c/eps [AT2] + 2 W^el_g).  A product of two trilinear functions
// has degree 2 per variable, so M_q depends on the q_g only through their 27
// moments
//   Q_pqr = sum_g q_g xi_g^p eta_g^q zeta_g^r / 64,  p, q, r <= 2,
// precomputed once per U (vfg_v_set_u): (M_q x)_abc = sum Q_(a+a',b+b',c+c') x_a'b'c'
// in modal sums (vfg_modal.h), 64 FMAs per element, and L is diagonal there.
#include "vfg_modal.h"
#include "vfg_kernels.h"

namespace vfg {

struct VConst {
  double ks[8];     // ks L in modal sums: c eps vol / 16 sum_d (1/h_d^2) (1/3)^(other powers)
  double crhs;      // Gc/atCv/eps * (.5 AT2 | .25 AT1), VFMech.c:2350-2384
};

// the launch constants are formed in extended precision and rounded once: a
// constant's error is the same in every element, so it does not average out
static VConst make_vconst(const DevProblem &P) {
  VConst C;
  const long double h[3] = {P.G.hx, P.G.hy, P.G.hz}, c = .5L * P.Gc / P.atcv;
  for (int i = 0; i < 8; i++) {
    long double t = 0.;
    for (int d = 0; d < 3; d++) {
      if (!um_pow(i, d)) continue;
      long double w = 1. / (h[d] * h[d]);
      for (int e = 0; e < 3; e++)
        if (e != d && um_pow(i, e)) w /= 3.;
      t += w;
    }
    C.ks[i] = (double)(c * P.eps * h[0] * h[1] * h[2] / 16. * t);
  }
  C.crhs = P.atnum == 2 ? P.Gc / P.atcv / P.eps * .5 : P.Gc / P.atcv / P.eps * .25;
  return C;
}

// -------------------------------------------------------------- setup: Vq
// launch constants: strains are formed times 4 hz, so that d_z takes the modal
// sums as they are
struct VSetup {
  double kx, ky;    // hz / hx, hz / hy
  double kth;       // alpha dtheta of a modal sum, times 4 hz
  double lam, mu2;  // lam, 2 mu for E = 1, over (4 hz)^2
  double cm, vol;   // AT2 mass term; vol / 64
};
static VSetup make_vsetup(const DevProblem &P) {
  const Grid &G = P.G;
  const long double s = 16.L * G.hz * G.hz;
  VSetup C;
  C.kx = G.hz / G.hx;
  C.ky = G.hz / G.hy;
  C.kth = P.alpha * G.hz / 2.;
  C.lam = (double)(P.lam1 / s);
  C.mu2 = (double)(2. * P.mu1 / s);
  C.cm = P.atnum == 2 ? (double)(.5L * P.Gc / P.atcv / P.eps) : 0.;
  C.vol = (double)((long double)G.hx * G.hy * G.hz / 64.);
  return C;
}

// One block per (tile, element layer), one thread per tile slot: element
// (15 bx - 1 + tx, 15 by - 1 + ty) of the V operator's tile-blocked layout
// (halo elements are computed by every tile that holds them), so each
// coefficient is written as one aligned, contiguous 512-byte segment per
// wavefront.  The strains at the Gauss points come from the modal sums of the
// corners; the moments are summed row by row.
// UNI: UNILATERAL_NOCOMPRESSION (VFMech.c:183-208, 2125-2153), 1/2 sigma(eps -
// e0) : eps, less kappa tr^2 / 2 where tr(eps) < 0.
// Bound by issue and the write of the moments, which do not overlap (128^3:
// about 105 us without the stores, 79 us for a fill of their 515 MB): about 950
// FP64 operations per element against 2400 interpolating values and gradients
// at each point; 128^3 187 -> 173 us.  Staging the node planes in LDS over
// several layers, or storing each third of the moments when complete, is no
// faster (164 us, and the apply after it loses as much to the caches).
template <bool UNI>
__global__ __launch_bounds__(256, 2) void k_v_setup(DevProblem P, VSetup C, const double *__restrict__ U) {
  const Grid &G = P.G;
  const int tid = threadIdx.x;
  const Blk3 b = xcd_block();
  const int ei = b.x * 15 - 1 + tid % 16, ej = b.y * 15 - 1 + tid / 16, ek = b.z;
  const int tile = b.x + gridDim.x * b.y;
  double *out = P.Vq + tiled_index(tile, ek, G.nez, 27, tid);
  if (ei < 0 || ei >= G.nex || ej < 0 || ej >= G.ney) {
    for (int g = 0; g < 27; g++) out[g * 64] = 0.;
    return;
  }
  double M[3][8], Th[8];  // modal sums of u_c and of alpha dtheta
  {
    double fld[4][8];
#pragma unroll
    for (int a = 0; a < 8; a++) {
      const int64_t n = node_id(G, ei + (a & 1), ej + ((a >> 1) & 1), ek + (a >> 2));
#pragma unroll
      for (int c = 0; c < 3; c++) fld[c][a] = U[3 * n + c];
      fld[3][a] = P.dth[n];
    }
#pragma unroll
    for (int c = 0; c < 3; c++) modal_sums([&](int a) { return fld[c][a]; }, M[c]);
    modal_sums([&](int a) { return fld[3][a]; }, Th);
  }
  const double Ee = P.E_elem ? P.E_elem[cell_id(G, ei, ej, ek)] : P.E;
  const double lam = C.lam * Ee, mu2 = C.mu2 * Ee, kap = lam + mu2 * (1. / 3.);
#pragma unroll
  for (int q = 0; q < 8; q++) Th[q] *= C.kth;
  constexpr double X1 = VFG_SQ35, X2 = .6;  // Gauss point +1 and its square (point -1: -X1; the middle one 0)
  double Q[3][3][3];                        // [r][q][p]
#pragma unroll
  for (int q = 0; q < 9; q++)
#pragma unroll
    for (int r = 0; r < 3; r++) Q[r][q / 3][q % 3] = 0.;
#pragma unroll
  for (int gz = 0; gz < 3; gz++) {
    double dx[3][2], dy[3][3], th[4], Y[3][3];  // Y: [q][p] of the layer
#pragma unroll
    for (int c = 0; c < 3; c++) {
#pragma unroll
      for (int q = 0; q < 2; q++) dx[c][q] = C.kx * at_gauss(gz, M[c][1 + 2 * q], M[c][5 + 2 * q]);
      const double y0 = C.ky * at_gauss(gz, M[c][2], M[c][6]), y1 = C.ky * at_gauss(gz, M[c][3], M[c][7]);
#pragma unroll
      for (int gx = 0; gx < 3; gx++) dy[c][gx] = at_gauss(gx, y0, y1);
#pragma unroll
      for (int p = 0; p < 3; p++) Y[c][p] = 0.;
    }
#pragma unroll
    for (int q = 0; q < 4; q++) th[q] = at_gauss(gz, Th[q], Th[q + 4]);
#pragma unroll
    for (int gy = 0; gy < 3; gy++) {
      double hx[3], z0[3], z1[3], row[3];
#pragma unroll
      for (int c = 0; c < 3; c++) {
        hx[c] = at_gauss(gy, dx[c][0], dx[c][1]);
        z0[c] = at_gauss(gy, M[c][4], M[c][6]);
        z1[c] = at_gauss(gy, M[c][5], M[c][7]);
      }
      const double th0 = at_gauss(gy, th[0], th[2]), th1 = at_gauss(gy, th[1], th[3]);
#pragma unroll
      for (int gx = 0; gx < 3; gx++) {
        const double t = at_gauss(gx, th0, th1), f11 = hx[0], f22 = dy[1][gx], f33 = at_gauss(gx, z0[2], z1[2]);
        const double t01 = dy[0][gx] + hx[1], t02 = at_gauss(gx, z0[0], z1[0]) + hx[2],
                     t12 = at_gauss(gx, z0[1], z1[1]) + dy[2][gx];
        const double e11 = f11 - t, e22 = f22 - t, e33 = f33 - t, tr = (e11 + e22) + e33;
        const double sh = .5 * (t01 * t01 + t02 * t02 + t12 * t12);
        double W2;  // 2 W
        if constexpr (UNI) {
          const double trf = (f11 + f22) + f33;
          W2 = C.cm + lam * (tr * trf) + mu2 * (sh + (e11 * f11 + e22 * f22 + e33 * f33));
          if (trf < 0.) W2 -= kap * (trf * trf);
        } else {
          W2 = C.cm + lam * (tr * tr) + mu2 * (sh + (e11 * e11 + e22 * e22 + e33 * e33));
        }
        row[gx] = gW(gx) * W2;
      }
      const double S = row[0] + row[2], w = C.vol * gW(gy) * gW(gz);
      const double m[3] = {w * (S + row[1]), (w * X1) * (row[2] - row[0]), (w * X2) * S};
#pragma unroll
      for (int p = 0; p < 3; p++) {
        Y[0][p] += m[p];
        if (gy != 1) {
          Y[1][p] += gy ? X1 * m[p] : -X1 * m[p];
          Y[2][p] += X2 * m[p];
        }
      }
    }
#pragma unroll
    for (int q = 0; q < 3; q++)
#pragma unroll
      for (int p = 0; p < 3; p++) {
        Q[0][q][p] += Y[q][p];
        if (gz != 1) {
          Q[1][q][p] += gz ? X1 * Y[q][p] : -X1 * Y[q][p];
          Q[2][q][p] += X2 * Y[q][p];
        }
      }
  }
#pragma unroll
  for (int r = 0; r < 3; r++)
#pragma unroll
    for (int q = 0; q < 3; q++)
#pragma unroll
      for (int p = 0; p < 3; p++) out[((r * 3 + q) * 3 + p) * 64] = Q[r][q][p];
}

int64_t vq_doubles(const Grid &G) {
  return (int64_t)((G.nx + 14) / 15) * ((G.ny + 14) / 15) * G.nez * 27 * 256;
}

__global__ void k_v_fixmask(DevProblem P) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= P.nn) return;
  const Grid &G = P.G;
  int i = (int)(n % G.nx), j = (int)((n / G.nx) % G.ny), k = (int)(n / ((int64_t)G.nx * G.ny));
  bool f = on_dirichlet(G, P.bcV.face[0], P.bcV.vert[0], i, j, k);
  if (P.atnum == 2 && P.VIrrev[n] <= P.irrevtol) f = true;  // VF_IrrevApplyEQMat
  P.vfix[n] = f ? 1 : 0;
}

// ------------------------------------------------------------------- apply
// the 27 moments of one element, read one layer ahead by the march
struct VQ {
  double q[27];  // [r][q][p]
};
// the parts of the march's interface that the V operators share: one nodal
// field, the moments of the tile-blocked layout
struct VModBase {
  using T = double;
  static constexpr int NF = 1, NC = 1;
  struct Face {
    double m[4], own;  // modal sums of the face; the thread's own node
  };
  struct Own {
    double x;
  };
  using Aux = VQ;
  const double *q;
  const uint8_t *vfix;
  Grid G;
  VConst C;
  template <class RD>
  __device__ void face(const RD &rd, Face &F) const {
    const double x0 = rd(0, 0), x1 = rd(0, 1), x2 = rd(0, 2), x3 = rd(0, 3);
    const double a = x0 + x1, b = x2 + x3, e = x1 - x0, f = x3 - x2;
    F.m[0] = a + b;
    F.m[1] = e + f;
    F.m[2] = b - a;
    F.m[3] = f - e;
    F.own = x3;
  }
  __device__ Own own(const Face &F) const { return Own{F.own}; }
  // NT: streamed past the caches
  template <bool NT>
  __device__ VQ moments(int ek, int tile, int slot) const {
    VQ a;
    const double *b = q + tiled_index(tile, ek, G.nez, 27, 0);  // uniform in the workgroup
#pragma unroll
    for (int g = 0; g < 27; g++) {
      const double *p = b + g * 64 + (unsigned)(slot / 64 * (27 * 64) + slot % 64);
      a.q[g] = NT ? __builtin_nontemporal_load(p) : *p;
    }
    return a;
  }
  __device__ VQ aux(int, int, int ek, int tile, int slot) const { return moments<false>(ek, tile, slot); }
};
// adds the modal forces y[8] of a layer to the planes below and above it
__device__ __forceinline__ void v_planes(const double (&y)[8], double (&tot)[1][4], double (&carry)[1][4]) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    tot[0][i] += y[i] - y[i + 4];
    carry[0][i] = y[i] + y[i + 4];
  }
}

// an owned node's data, read a layer before its store: a load issued there
// would wait for the next layer's moments, which are in flight by then
struct VOwn {
  double x, b, irr;
  uint8_t fix;
};
// MODE 0: masked Jacobian; 1: VF_VResidual; 2: plain K x
struct VApplyRec : VModBase {
  const double *x;
  double *y;
  const double *bV, *VIrrev;
  BcMask bc;
  uint8_t ftype[6], vtype[8];
  int atnum;
  double irrevtol;
};
struct VRaw {
  double x;
  uint8_t fix;
};
template <int MODE>
struct VApplyOp : VApplyRec {
  using Raw = VRaw;
  static __device__ VRaw off() { return VRaw{0., 1}; }
  __device__ VRaw load(int, int64_t n) const { return VRaw{x[n], MODE == 0 ? vfix[n] : (uint8_t)0}; }
  __device__ double stage(int, const VRaw &r) const { return r.fix ? 0. : r.x; }
  __device__ VOwn own_load(int64_t n) const {
    VOwn o{};
    if constexpr (MODE == 0) {
      o.fix = vfix[n];
      o.x = x[n];
    }
    if constexpr (MODE == 1) {
      o.b = bV[n];
      if (atnum == 2) o.irr = VIrrev[n];
    }
    return o;
  }
  __device__ void element(const VQ &Q, const Face &B, const Face &F, double (&tot)[1][4], double (&carry)[1][4]) const {
    double X[8], R[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      X[i] = B.m[i] + F.m[i];
      X[i + 4] = F.m[i] - B.m[i];
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
      R[i] = C.ks[i] * X[i];
#pragma unroll
      for (int j = 0; j < 8; j++)
        R[i] += Q.q[(um_pow(i, 0) + um_pow(j, 0)) + 3 * (um_pow(i, 1) + um_pow(j, 1)) +
                    9 * (um_pow(i, 2) + um_pow(j, 2))] * X[j];
    }
    v_planes(R, tot, carry);
  }
  __device__ void store(int64_t n, uint32_t fb, const double (&acc)[1], const Own &own, const VOwn &o) const {
    if constexpr (MODE == 0) {
      y[n] = o.fix ? o.x : acc[0];
    } else if constexpr (MODE == 2) {
      y[n] = acc[0];
    } else {
      // VF_VResidual: F = K V - b; AT2 irreversible rows -> 0 (VF_IrrevApplyEQVec);
      // then ResidualApplyDirichletBC with V as its own BC vector.
      double F = acc[0] - o.b;
      if (atnum == 2 && o.irr <= irrevtol) F = 0.;
      if (face_dirichlet(bc.face[0], bc.vert[0], fb)) {
        int t = 0;
        for (int f = 0; f < 6; f++)
          if (ftype[f] && (fb >> f & 1u)) t = ftype[f];
        const int v = face_vertex(fb);
        if (v >= 0 && vtype[v]) t = vtype[v];
        F = t == 2 ? own.x - 1. : t == 3 ? 0. : own.x;
      }
      y[n] = F;
    }
  }
};

// CG-fused masked apply: stages p = z + beta p_old off the mask, writes
// p and q = K p, one partial of p.q per workgroup; p_old (x) and p are different
// arrays (neighbouring workgroups still read p_old at their halo nodes)
struct VApplyCgOp : VApplyOp<0> {
  const double *z;
  double *pw;
  double *part;
  double bval;  // beta, formed by the kernel
  struct Raw {
    double z, x;
    uint8_t fix;
  };
  static __device__ Raw off() { return Raw{0., 0., 1}; }
  __device__ Raw load(int, int64_t n) const { return Raw{z[n], x[n], vfix[n]}; }
  __device__ double stage(int, const Raw &r) const { return r.fix ? 0. : r.z + bval * r.x; }
  __device__ uint8_t own_load(int64_t n) const { return vfix[n]; }
  __device__ double store(int64_t n, uint32_t, const double (&acc)[1], const Own &own, uint8_t fix) const {
    const double yv = fix ? own.x : acc[0];
    y[n] = yv;
    pw[n] = own.x;
    return own.x * yv;
  }
  __device__ void partial(int slot, double v) const { part[slot] = v; }
};

// Bound by the read of the moments (216 B per element, 1.27 x with the halo
// slots at 128^3): 128^3 120 us = 5.1 TB/s, 141 us for the 27 Gauss weights read
// a plane at a time.  All 27 of the next layer are in flight during a layer;
// the 176 registers that takes leave two waves per SIMD (three spill: 151 us).
// NT: a moment array well over the 256 MB last-level cache is streamed past it,
// one that fits is kept there for the next product.  Kept and streamed, back to
// back, 105 x 105 nodes by 60 to 220 elements: 163 MB 33.4 and 38.8 us, 284 MB 55.3
// and 65.7, 325 MB 70.6 and 72.5, 352 MB 80.3 and 79.7, 406 MB 90.8 and 88.8, 515 MB
// 118.5 and 111.1, 596 MB 137.3 and 128.2.  They cross near 340 MB; up to the line
// the choice loses 2 % at most.
constexpr int64_t V_STREAM_BYTES = 400ll << 20;
template <int MODE, bool NT>
struct VApplyStreamOp : VApplyOp<MODE> {
  __device__ VQ aux(int, int, int ek, int tile, int slot) const { return this->template moments<NT>(ek, tile, slot); }
};
template <int MODE, bool NT>
__global__ __launch_bounds__(256, 2) void k_v_apply(VApplyStreamOp<MODE, NT> op, int OZ) {
  march_modal<16, 16>(op.G, op, OZ, xcd_block());
}

// The same over a list of workgroups.  The reduced Newton systems of the
// V-solve live on the free nodes, a thin band around the cracks: a workgroup
// owning no free node has p = q = 0 throughout and is left out.  The list
// (k_v_list_chunks) holds chunk ids tile + txy * zc, a chunk being the node
// planes [zc L, zc L + L) of a 15 x 15 node tile; L sits in list[cap + 1].
// Partials are written compactly, one per list entry.
struct VChunk {
  int bx, by, bz, L;
};
__device__ __forceinline__ VChunk chunk_at(const Grid &G, const int *__restrict__ list, int cap, int w) {
  const int gx = (G.nx + 14) / 15, txy = gx * ((G.ny + 14) / 15);
  const int c = __builtin_amdgcn_readfirstlane(list[w]), t = c % txy;  // uniform: the moments' base address too
  return VChunk{t % gx, t / gx, c / txy, __builtin_amdgcn_readfirstlane(list[cap + 1])};
}
// the sums of n pairs, or of n values in the first of them, in every thread
template <int W>
__device__ __forceinline__ void vcg_sums(const double *__restrict__ part, int n, double (&s)[W]) {
  __shared__ double sh[4], bc[W];
  double a[W] = {};
  for (int i = threadIdx.x; i < n; i += 256)
#pragma unroll
    for (int w = 0; w < W; w++) a[w] += part[W * i + w];
#pragma unroll
  for (int w = 0; w < W; w++) {
    const double v = block_sum<256>(a[w], sh);
    if (threadIdx.x == 0) bc[w] = v;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < W; w++) s[w] = bc[w];
}
// group b of the output sums the b-th part of the n groups
template <int W>
__global__ __launch_bounds__(256) void k_vcg_fold(const double *__restrict__ part, int n, double *__restrict__ out) {
  const int per = (n + VCG_FOLD - 1) / VCG_FOLD, lo = blockIdx.x * per, hi = lo + per < n ? lo + per : n;
  double s[W];
  vcg_sums<W>(part + (int64_t)W * lo, hi - lo, s);
  if (threadIdx.x == 0)
#pragma unroll
    for (int w = 0; w < W; w++) out[W * blockIdx.x + w] = s[w];
}
__global__ __launch_bounds__(256, 2) void k_v_apply_cg_list(VApplyCgOp op, const int *__restrict__ list, int cap,
                                                           VCgStep c) {
  // the CG has converged: read by one thread, since the first workgroup may set it
  // meanwhile (below) and a workgroup has to leave or stay as a whole
  __shared__ int done;
  if (threadIdx.x == 0) done = c.sc[S_DONE] != 0.;
  __syncthreads();
  if (done) return;
  double s[2];
  vcg_sums<2>(c.pairs, c.npairs, s);
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  if (c.k > 0 && c.tol2 > 0. && s[1] <= c.tol2) {  // in every workgroup alike
    if (first) {
      c.sc[S_DONE] = 1.;
      c.sc[S_RR] = s[1];
      c.sc[S_ITS] = (double)c.k;
    }
    return;
  }
  const double old = c.sc[S_RZ];
  op.bval = c.k > 0 && old != 0. ? s[0] / old : 0.;
  if (first) {
    c.sc[S_RZ1] = s[0];
    if (!isfinite(s[0]) || !isfinite(s[1])) c.sc[S_FLAG] = 2.;
  }
  const VChunk q = chunk_at(op.G, list, cap, blockIdx.x);
  march_modal<16, 16>(op.G, op, q.L, q.bx, q.by, q.bz, blockIdx.x);
}
// the plain apply over the listed chunks
template <int MODE>
__global__ __launch_bounds__(256, 2) void k_v_apply_list(VApplyOp<MODE> op, const int *__restrict__ list, int cap) {
  const VChunk q = chunk_at(op.G, list, cap, blockIdx.x);
  march_modal<16, 16>(op.G, op, q.L, q.bx, q.by, q.bz);
}

__global__ void k_fill_u32(uint32_t *a, uint32_t v, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = v;
}

// flag[tile + txy k] = 1 where node plane k of a 15 x 15 node tile holds a
// node with mask == 0 (flag cleared beforehand)
__global__ void k_v_mark_planes(Grid G, const uint8_t *__restrict__ mask, uint32_t *__restrict__ flag) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (int64_t)G.nx * G.ny * G.nz || mask[n]) return;
  const int i = (int)(n % G.nx), j = (int)((n / G.nx) % G.ny), k = (int)(n / ((int64_t)G.nx * G.ny));
  const int gx = (G.nx + 14) / 15, txy = gx * ((G.ny + 14) / 15);
  flag[i / 15 + gx * (j / 15) + (int64_t)txy * k] = 1u;  // same value from every writer
}

// out[tile + txy k] = 1 where a flag is set on one of the 3 x 3 tiles around
// the tile, on planes k - 1 .. k + 1: the (tile, plane) pairs holding a node
// that shares an element with a node of a flagged pair (a node at a tile edge
// meets the next tile's nodes, a node plane the planes next to it)
__global__ void k_v_dilate_planes(const uint32_t *__restrict__ in, uint32_t *__restrict__ out, int gx, int gy,
                                  int nz) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t txy = (int64_t)gx * gy;
  if (f >= txy * nz) return;
  const int t = (int)(f % txy), k = (int)(f / txy), tx = t % gx, ty = t / gx;
  uint32_t any = 0u;
  for (int dk = -1; dk <= 1; dk++) {
    const int kk = k + dk;
    if (kk < 0 || kk >= nz) continue;
    for (int dy = -1; dy <= 1; dy++) {
      const int yy = ty + dy;
      if (yy < 0 || yy >= gy) continue;
      for (int dx = -1; dx <= 1; dx++) {
        const int xx = tx + dx;
        if (xx >= 0 && xx < gx) any |= in[xx + (int64_t)gx * yy + txy * kk];
      }
    }
  }
  out[f] = any ? 1u : 0u;
}

constexpr int VLT = 1024;  // threads of the chunk-list kernel

__device__ __forceinline__ int block_isum(int v, int *sh) {
  __syncthreads();
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int o = VLT / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
    __syncthreads();
  }
  return sh[0];
}

// One workgroup of VLT threads.  Chunk length L = ceil(flagged planes /
// target), clamped to [lmin, lmax]: a thin band gives many one-plane chunks
// (latency, not work, bounds the march of a few chunks), a wide one long
// chunks (each chunk re-reads one halo plane).  The flagged chunks are listed
// in increasing id; list[cap] = their count, list[cap + 1] = L.
__global__ __launch_bounds__(VLT) void k_v_list_chunks(const uint32_t *__restrict__ flag, int txy, int nz, int lmin,
                                                       int lmax, int target, int *__restrict__ list, int cap) {
  __shared__ int sh[VLT];
  const int tid = threadIdx.x;
  const int64_t nf = (int64_t)txy * nz;
  int f = 0;
  for (int64_t i = tid; i < nf; i += VLT) f += flag[i] != 0u;
  const int F = block_isum(f, sh);
  int L = (F + target - 1) / target;
  L = L < lmin ? lmin : L > lmax ? lmax : L;
  if (L < 1) L = 1;
  const int nzc = (nz + L - 1) / L;
  const int64_t nch = (int64_t)txy * nzc, per = (nch + VLT - 1) / VLT;
  const int64_t c0 = tid * per < nch ? tid * per : nch, c1 = c0 + per < nch ? c0 + per : nch;
  auto hit = [&](int64_t c) {
    const int t = (int)(c % txy), k0 = (int)(c / txy) * L, k1 = k0 + L < nz ? k0 + L : nz;
    for (int k = k0; k < k1; k++)
      if (flag[t + (int64_t)txy * k]) return true;
    return false;
  };
  int cnt = 0;
  for (int64_t c = c0; c < c1; c++) cnt += hit(c);
  // exclusive scan of the per-thread counts
  __syncthreads();
  sh[tid] = cnt;
  __syncthreads();
  for (int o = 1; o < VLT; o <<= 1) {
    const int v = tid >= o ? sh[tid - o] : 0;
    __syncthreads();
    sh[tid] += v;
    __syncthreads();
  }
  int off = sh[tid] - cnt;
  for (int64_t c = c0; c < c1; c++)
    if (hit(c)) list[off++] = (int)c;
  if (tid == VLT - 1) {
    list[cap] = sh[VLT - 1];
    list[cap + 1] = L;
  }
}

// x += alpha p, r -= alpha q, z = dinv r and the partials of r.z, r.r over
// the owned nodes of the listed chunks (p = q = r = 0 elsewhere)
__global__ __launch_bounds__(256) void k_v_xr_list(Grid G, const int *__restrict__ list, int cap,
                                                   double *__restrict__ x, double *__restrict__ r,
                                                   double *__restrict__ z, const double *__restrict__ p,
                                                   const double *__restrict__ q, const double *__restrict__ dinv,
                                                   const double *__restrict__ ppq, int npq, double *__restrict__ part,
                                                   VCgStep cg) {
  if (cg.sc[S_DONE] != 0.) return;  // the CG has converged
  __shared__ double sh[4];
  const int gx = (G.nx + 14) / 15, txy = gx * ((G.ny + 14) / 15);
  const int c = list[blockIdx.x], L = list[cap + 1], t = c % txy;
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int i = (t % gx) * 15 + tx, j = (t / gx) * 15 + ty, k0 = (c / txy) * L;
  const int k1 = k0 + L < G.nz ? k0 + L : G.nz;
  double pq[1];
  vcg_sums<1>(ppq, npq, pq);
  const bool ok = pq[0] > 0. && isfinite(pq[0]);
  const double old = cg.sc[S_RZ1], al = ok ? old / pq[0] : 0.;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    cg.sc[S_RZ] = old;
    if (!ok) cg.sc[S_FLAG] = isfinite(pq[0]) ? 1. : 2.;
  }
  double rz = 0., rr = 0.;
  if (tx < 15 && ty < 15 && i < G.nx && j < G.ny)
    for (int k = k0; k < k1; k++) {
      const int64_t n = node_id(G, i, j, k);
      x[n] += al * p[n];
      const double ri = r[n] - al * q[n];
      r[n] = ri;
      const double zi = dinv[n] * ri;
      z[n] = zi;
      rz += ri * zi;
      rr += ri * ri;
    }
  rz = block_sum<256>(rz, sh);
  rr = block_sum<256>(rr, sh);
  if (threadIdx.x == 0) { part[2 * blockIdx.x] = rz; part[2 * blockIdx.x + 1] = rr; }
}

// ---------------------------------------------------------------- diagonal
// d_a = sum over modal pairs of signs times Q and ks: per direction
// Q_0 + 2 s Q_1 + Q_2 with s = -1, 1 the corner's side
struct VDiagOp : VModBase {
  double *d;
  using Raw = double;
  static __device__ double off() { return 0.; }
  __device__ double load(int, int64_t) const { return 0.; }
  __device__ double stage(int, double v) const { return v; }
  __device__ void element(const VQ &Q, const Face &, const Face &, double (&tot)[1][4], double (&carry)[1][4]) const {
    double a[3][3][2], b[3][2][2], r[2][2][2], L = 0.;
#pragma unroll
    for (int i = 0; i < 8; i++) L += C.ks[i];
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int j = 0; j < 3; j++) {
        const double *m = Q.q + (k * 3 + j) * 3;
        const double S = m[0] + m[2];
        a[k][j][0] = S - 2. * m[1];
        a[k][j][1] = S + 2. * m[1];
      }
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const double S = a[k][0][i] + a[k][2][i];
        b[k][0][i] = S - 2. * a[k][1][i];
        b[k][1][i] = S + 2. * a[k][1][i];
      }
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const double S = b[0][j][i] + b[2][j][i];
        r[0][j][i] = L + (S - 2. * b[1][j][i]);
        r[1][j][i] = L + (S + 2. * b[1][j][i]);
      }
    // the corner values as modal sums of the two faces
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const double s0 = .25 * (r[k][0][0] + r[k][0][1]), s1 = .25 * (r[k][1][0] + r[k][1][1]);
      const double e0 = .25 * (r[k][0][1] - r[k][0][0]), e1 = .25 * (r[k][1][1] - r[k][1][0]);
      double(&o)[4] = k ? carry[0] : tot[0];
      const double m[4] = {s0 + s1, e0 + e1, s1 - s0, e1 - e0};
#pragma unroll
      for (int q = 0; q < 4; q++) o[q] = k ? m[q] : o[q] + m[q];
    }
  }
  __device__ uint8_t own_load(int64_t n) const { return vfix[n]; }
  __device__ void store(int64_t n, uint32_t, const double (&acc)[1], const Own &, uint8_t fix) const {
    d[n] = fix ? 1. : acc[0];
  }
};

__global__ __launch_bounds__(256, 2) void k_v_diag(VDiagOp op, int OZ) { march_modal<16, 16>(op.G, op, OZ, xcd_block()); }
__global__ __launch_bounds__(256, 2) void k_v_diag_list(VDiagOp op, const int *__restrict__ list, int cap) {
  const VChunk q = chunk_at(op.G, list, cap, blockIdx.x);
  march_modal<16, 16>(op.G, op, q.L, q.bx, q.by, q.bz);
}

// ------------------------------------------------------------ load vector
// b_a = crhs sum_g W phi_a + [pressurize] sum_g W p (u . grad phi_a)
// In modal duals R: R_0 = crhs vol / 8 (the rule integrates phi_a exactly) and,
// for the modes i with variable d, R_i += vol / (4 h_d) <p u_d mono_i / x_d> in
// closed form.
// About 230 FP64 operations per element, against 700 of a walk over the Gauss
// points; 97 x 131 x 76 39 -> 23 us (near the read of U and p).
struct VRhsOp {
  using T = double;
  static constexpr int NF = 4, NC = 1;
  const double *U, *p;
  double *b;
  Grid G;
  double at, kf[3];  // crhs vol / 8; vol / (256 h_d)
  int crack;
  struct Face {
    double f[4][4];  // u_c, p: s, x, y, w
  };
  struct Own {};
  struct Aux {};
  using Raw = double;
  static __device__ double off() { return 0.; }
  __device__ double load(int f, int64_t n) const { return f < 3 ? U[3 * n + f] : p[n]; }
  __device__ double stage(int, double x) const { return x; }
  template <class RD>
  __device__ void face(const RD &rd, Face &F) const {
#pragma unroll
    for (int f = 0; f < 4; f++) {
      const double x0 = rd(f, 0), x1 = rd(f, 1), x2 = rd(f, 2), x3 = rd(f, 3);
      const double s0 = x0 + x1, s1 = x2 + x3, d0 = x1 - x0, d1 = x3 - x2;
      F.f[f][0] = s0 + s1;
      F.f[f][1] = d0 + d1;
      F.f[f][2] = s1 - s0;
      F.f[f][3] = d1 - d0;
    }
  }
  __device__ Own own(const Face &) const { return Own{}; }
  __device__ Aux aux(int, int, int, int, int) const { return Aux{}; }
  __device__ void element(const Aux &, const Face &B, const Face &F, double (&tot)[1][4], double (&carry)[1][4]) const {
    double R[8] = {at, 0., 0., 0., 0., 0., 0., 0.};
    if (crack) {
      double Pm[8], Um[3][8];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        Pm[q] = F.f[3][q] + B.f[3][q];
        Pm[q + 4] = F.f[3][q] - B.f[3][q];
#pragma unroll
        for (int c = 0; c < 3; c++) {
          Um[c][q] = F.f[c][q] + B.f[c][q];
          Um[c][q + 4] = F.f[c][q] - B.f[c][q];
        }
      }
#pragma unroll
      for (int d = 0; d < 3; d++) {
        double M[2][2][2];  // by the power of variable d in p and u
#pragma unroll
        for (int t = 0; t < 2; t++) {
          double p2[2][2], u2[2][2];
#pragma unroll
          for (int q = 0; q < 4; q++) {
            p2[q & 1][q >> 1] = Pm[modal_at(d, t, q & 1, q >> 1)];
            u2[q & 1][q >> 1] = Um[d][modal_at(d, t, q & 1, q >> 1)];
          }
          bilinear_moments(p2, u2, M[t]);
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int i = q & 1, j = q >> 1;
          R[modal_at(d, 1, i, j)] += (kf[d] * (i + j == 2 ? 1. / 9. : i + j ? 1. / 3. : 1.)) *
                                     (M[0][i][j] + (1. / 3.) * M[1][i][j]);
        }
      }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      tot[0][q] += R[q] - R[q + 4];
      carry[0][q] = R[q] + R[q + 4];
    }
  }
  __device__ void store(int64_t n, uint32_t, const double (&acc)[1], const Own &) const { b[n] = acc[0]; }
};

__global__ __launch_bounds__(256, 2) void k_v_rhs(VRhsOp op, int OZ) { march_modal<16, 16>(op.G, op, OZ, xcd_block()); }

// ------------------------------------------------------------ launchers
static dim3 mgrid(const Grid &G, int OZ) {
  return dim3((G.nx + 14) / 15, (G.ny + 14) / 15, (G.nz + OZ - 1) / OZ);
}
int choose_oz(const Grid &G, int tiles_xy, int slots);
// z-chunk length of the V kernels: whole rounds of resident workgroups, as for
// the u kernels; a partial last round costs a full one
int device_slots_of(const void *kernel, int threads);
static int v_slots() {
  static int n = device_slots_of((const void *)k_v_apply<0, false>, 256);
  return n;
}
static int oz_for(const Grid &G) { return choose_oz(G, ((G.nx + 14) / 15) * ((G.ny + 14) / 15), v_slots()); }

void launch_v_setup(const DevProblem &P, const double *U, hipStream_t s) {
  VRhsOp op;
  op.U = U; op.p = P.p; op.b = P.bV; op.G = P.G;
  const double h[3] = {P.G.hx, P.G.hy, P.G.hz}, vol = h[0] * h[1] * h[2];
  op.at = make_vconst(P).crhs * vol / 8.;
  for (int d = 0; d < 3; d++) op.kf[d] = vol / (256. * h[d]);
  op.crack = P.hasCrackPressure;
  int OZ = oz_for(P.G);
  hipLaunchKernelGGL(k_v_rhs, mgrid(P.G, OZ), dim3(256), 0, s, op, OZ);
  // after the load: the moments are what the next product reads, and the last written
  const dim3 g((P.G.nx + 14) / 15, (P.G.ny + 14) / 15, P.G.nez);
  if (P.unilateral) hipLaunchKernelGGL(k_v_setup<true>, g, dim3(256), 0, s, P, make_vsetup(P), U);
  else hipLaunchKernelGGL(k_v_setup<false>, g, dim3(256), 0, s, P, make_vsetup(P), U);
}

void launch_v_fixmask(const DevProblem &P, hipStream_t s) {
  hipLaunchKernelGGL(k_v_fixmask, dim3((unsigned)((P.nn + 255) / 256)), dim3(256), 0, s, P);
}

static void v_fill(VModBase &op, const DevProblem &P, const uint8_t *mask) {
  op.q = P.Vq;
  op.vfix = mask ? mask : P.vfix;
  op.G = P.G;
  op.C = make_vconst(P);
}
static void vapply_fill(VApplyRec &op, const DevProblem &P, const double *x, double *y, const uint8_t *mask) {
  v_fill(op, P, mask);
  op.x = x; op.y = y; op.bV = P.bV; op.VIrrev = P.VIrrev; op.bc = P.bcV;
  for (int f = 0; f < 6; f++) op.ftype[f] = (uint8_t)P.hbcV.face[f];
  for (int v = 0; v < 8; v++) op.vtype[v] = (uint8_t)P.hbcV.vertex[v];
  op.atnum = P.atnum; op.irrevtol = P.irrevtol;
}
template <class Op>
static Op vapply_op(const VApplyRec &r) {
  Op op;
  static_cast<VApplyRec &>(op) = r;
  return op;
}
template <int MODE>
static void launch_v_apply_m(const VApplyRec &r, const dim3 &g, int OZ, bool stream, hipStream_t s) {
  if (stream)
    hipLaunchKernelGGL((k_v_apply<MODE, true>), g, dim3(256), 0, s, (vapply_op<VApplyStreamOp<MODE, true>>(r)), OZ);
  else
    hipLaunchKernelGGL((k_v_apply<MODE, false>), g, dim3(256), 0, s, (vapply_op<VApplyStreamOp<MODE, false>>(r)), OZ);
}

void launch_v_apply(const DevProblem &P, const double *x, double *y, int mode, hipStream_t s,
                    const uint8_t *mask) {
  VApplyRec r;
  vapply_fill(r, P, x, y, mask);
  const int OZ = oz_for(P.G);
  const dim3 g = mgrid(P.G, OZ);
  const bool stream = 8 * vq_doubles(P.G) > V_STREAM_BYTES;
  if (mode == 0) launch_v_apply_m<0>(r, g, OZ, stream, s);
  else if (mode == 1) launch_v_apply_m<1>(r, g, OZ, stream, s);
  else launch_v_apply_m<2>(r, g, OZ, stream, s);
}

void launch_v_apply_list(const DevProblem &P, const double *x, double *y, int mode, const int *list, int count,
                         hipStream_t s, const uint8_t *mask) {
  if (count <= 0) return;
  VApplyRec r;
  vapply_fill(r, P, x, y, mask);
  const dim3 g((unsigned)count);
  const int cap = v_chunk_cap(P.G);
  if (mode == 0) hipLaunchKernelGGL(k_v_apply_list<0>, g, dim3(256), 0, s, vapply_op<VApplyOp<0>>(r), list, cap);
  else if (mode == 1) hipLaunchKernelGGL(k_v_apply_list<1>, g, dim3(256), 0, s, vapply_op<VApplyOp<1>>(r), list, cap);
  else hipLaunchKernelGGL(k_v_apply_list<2>, g, dim3(256), 0, s, vapply_op<VApplyOp<2>>(r), list, cap);
}

// ------------------------------------------------ persistent multi-problem apply
// Masked Jacobian applies of several problems in one launch (serving engine):
// a work list of (member, tile x, tile y, z-chunk); the item count lives on the
// device and members whose flags[p * fstride] is 0 are skipped.
struct BVApply {
  VApplyOp<0> op;
  int OZ;
};
__global__ __launch_bounds__(256, 2) void k_batch_v_apply(const BVApply *__restrict__ probs,
                                                       const BItem *__restrict__ items,
                                                       const int *__restrict__ dcount,
                                                       const double *__restrict__ flags, int fstride) {
  const int n = *dcount;
  for (int it = blockIdx.x; it < n; it += gridDim.x) {
    const BItem w = items[it];
    if (flags[(int64_t)w.p * fstride] == 0.) continue;  // uniform per block
    const VApplyOp<0> &op = probs[w.p].op;  // read in place: the record is large
    const int OZ = probs[w.p].OZ;
    __syncthreads();  // LDS of the previous item is free
    march_modal<16, 16>(op.G, op, OZ, w.bx, w.by, w.bz);
  }
}
size_t vop_bytes() { return sizeof(BVApply); }
int v_oz(const Grid &G) { return oz_for(G); }
int v_apply_slots() { return v_slots(); }
void make_vop(const DevProblem &P, const double *x, double *y, const uint8_t *mask, void *out) {
  BVApply *b = (BVApply *)out;
  vapply_fill(b->op, P, x, y, mask);
  b->OZ = oz_for(P.G);
}
void launch_engine_v_apply(const void *d_ops, const BItem *items, const int *dcount, int grid, const double *flags,
                           int fstride, hipStream_t s) {
  hipLaunchKernelGGL(k_batch_v_apply, dim3(grid), dim3(256), 0, s, (const BVApply *)d_ops, items, dcount, flags,
                     fstride);
}

static VApplyCgOp make_vcg_op(const DevProblem &P, const double *pold, double *p, const double *z, double *q,
                              double *part, const uint8_t *mask) {
  VApplyCgOp op;
  vapply_fill(op, P, pold, q, mask);
  op.z = z; op.pw = p; op.part = part;
  return op;
}

int v_chunk_cap(const Grid &G) { return ((G.nx + 14) / 15) * ((G.ny + 14) / 15) * G.nz; }

void launch_v_chunk_list(const DevProblem &P, const uint8_t *mask, uint32_t *flag, int *list, hipStream_t s) {
  const int cap = v_chunk_cap(P.G), txy = cap / P.G.nz;
  // at most 32768 + txy chunks, whatever the band: partials fit the reduction buffers
  const int lmin = (cap + 32767) / 32768;
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)((cap + 255) / 256)), dim3(256), 0, s, flag, 0u, (int64_t)cap);
  hipLaunchKernelGGL(k_v_mark_planes, dim3((unsigned)((P.nn + 255) / 256)), dim3(256), 0, s, P.G, mask, flag);
  hipLaunchKernelGGL(k_v_list_chunks, dim3(1), dim3(VLT), 0, s, (const uint32_t *)flag, txy, P.G.nz, lmin, P.G.nz,
                     1024, list, cap);
}

void launch_v_dilated_list(const DevProblem &P, const uint32_t *flag, uint32_t *flag2, int *list2, hipStream_t s) {
  const int cap = v_chunk_cap(P.G), gx = (P.G.nx + 14) / 15, gy = (P.G.ny + 14) / 15, txy = gx * gy;
  const int lmin = (cap + 32767) / 32768;
  hipLaunchKernelGGL(k_v_dilate_planes, dim3((unsigned)((cap + 255) / 256)), dim3(256), 0, s, flag, flag2, gx, gy,
                     P.G.nz);
  hipLaunchKernelGGL(k_v_list_chunks, dim3(1), dim3(VLT), 0, s, (const uint32_t *)flag2, txy, P.G.nz, lmin, P.G.nz,
                     1024, list2, cap);
}

size_t vcg_partials(const Grid &G) {
  // launch_v_chunk_list: at most 32768 + one per tile
  const size_t cap = (size_t)v_chunk_cap(G), most = 32768 + cap / (size_t)G.nz, n = cap < most ? cap : most;
  return n < 2048 ? 2048 : n;
}

void launch_v_apply_cg_list(const DevProblem &P, const double *pold, double *p, const double *z, double *q, double *part,
                            const uint8_t *mask, const int *list, int count, const VCgStep &c, hipStream_t s) {
  if (count <= 0) return;
  const VApplyCgOp op = make_vcg_op(P, pold, p, z, q, part, mask);
  hipLaunchKernelGGL(k_v_apply_cg_list, dim3((unsigned)count), dim3(256), 0, s, op, list, v_chunk_cap(P.G), c);
}

void launch_v_xr_list(const Grid &G, const int *list, int count, double *x, double *r, double *z, const double *p,
                      const double *q, const double *dinv, const double *ppq, int npq, double *pairs, const VCgStep &c,
                      hipStream_t s) {
  if (count <= 0) return;
  hipLaunchKernelGGL(k_v_xr_list, dim3((unsigned)count), dim3(256), 0, s, G, list, v_chunk_cap(G), x, r, z, p, q,
                     dinv, ppq, npq, pairs, c);
}
void launch_vcg_fold(const double *part, int w, int n, double *out, hipStream_t s) {
  auto go = [&](auto k) { hipLaunchKernelGGL(k, dim3(VCG_FOLD), dim3(256), 0, s, part, n, out); };
  w == 2 ? go(k_vcg_fold<2>) : go(k_vcg_fold<1>);
}

void launch_v_diag(const DevProblem &P, double *d, hipStream_t s, const uint8_t *mask) {
  VDiagOp op;
  v_fill(op, P, mask);
  op.d = d;
  int OZ = oz_for(P.G);
  hipLaunchKernelGGL(k_v_diag, mgrid(P.G, OZ), dim3(256), 0, s, op, OZ);
}

void launch_v_diag_list(const DevProblem &P, double *d, const uint8_t *mask, const int *list, int count,
                        hipStream_t s) {
  if (count <= 0) return;
  VDiagOp op;
  v_fill(op, P, mask);
  op.d = d;
  hipLaunchKernelGGL(k_v_diag_list, dim3((unsigned)count), dim3(256), 0, s, op, list, v_chunk_cap(P.G));
}

}  // namespace vfg
