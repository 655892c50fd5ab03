// vfg_mg.hip -- geometric multigrid pieces for the u-solve preconditioner.
//
// The reference preconditions its u-CG with hypre BoomerAMG (PCHYPRE,
// VFCommon.c:1041-1047) on the assembled Jacobian; its large runs use PETSc
// GAMG with Chebyshev smoothers (-U_pc_type gamg, scripts/test16-*.sh).  On
// the structured grid of this path the same role is played matrix-free by
// geometric multigrid: about 2:1 coarsening of the element grid, coarse operators
// by rediscretisation, trilinear prolongation and its transpose.
//
//   level 1 coefficient of coarse element C: the mean of E_e * sbar_e over the
//     fine elements under C (weighted by overlap), sbar_e = sum_g w_g (v_g^2 +
//     eta) (weights summing to 1); level l+1 from level l likewise;
//   coarse operator: the Q1 elasticity operator with s = 1 and E = coefficient
//     (the u-apply with V = 1, eta = 0), so every level runs the same kernels.
// Dirichlet rows are excluded from restriction and prolongation on every
// level (their masks come from the same face/vertex table on each grid).
#include "vfg_internal.h"
#include "vfg_kernels.h"
#include "vfg_mg.h"
#include "vfg_modal.h"

namespace vfg {

// ------------------------------------------------------------ coefficients
// per fine element: E_e * sbar_e, sbar_e = sum_g w_g c_g with c_g = v_g^2 + eta,
// or, at the compressed points of a UNILATERAL_NOCOMPRESSION Jacobian (cmask),
// the factor that gives the isotropic coarse operator the point's P-wave
// modulus: c_g = (kappa (1 + eta) + 4/3 mu s_g) / (lam + 2 mu), kappa =
// lam + 2/3 mu (the spherical part there is not degraded)
// The mean of s = v^2 + eta over an element from the modal sums of v, orthogonal
// on it; UNI: at the Gauss points, compressed ones with their own weight.
template <bool UNI>
__global__ __launch_bounds__(256) void k_mg_elem_coef(Grid G, const double *__restrict__ V,
                                                      const double *__restrict__ E_elem, double E, double eta,
                                                      const uint32_t *__restrict__ cmask, double lam1, double mu1,
                                                      double *__restrict__ out) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)G.nex * G.ney * G.nez) return;
  const int ei = (int)(e % G.nex), ej = (int)((e / G.nex) % G.ney), ek = (int)(e / ((int64_t)G.nex * G.ney));
  double v[8], m[8];
#pragma unroll
  for (int a = 0; a < 8; a++) v[a] = V[node_id(G, ei + (a & 1), ej + ((a >> 1) & 1), ek + (a >> 2))];
  modal_sums([&](int a) { return v[a]; }, m);
  double s = 0.;
  if constexpr (UNI) {
    const uint32_t cm = cmask[e];
    const double kap1 = lam1 + 2. * mu1 / 3., pw = 1. / (lam1 + 2. * mu1);
#pragma unroll
    for (int gz = 0; gz < 3; gz++)
#pragma unroll
      for (int gy = 0; gy < 3; gy++) {
        double r[2];
#pragma unroll
        for (int x = 0; x < 2; x++)
          r[x] = at_gauss(gy, at_gauss(gz, m[x], m[x + 4]), at_gauss(gz, m[x + 2], m[x + 6]));
#pragma unroll
        for (int gx = 0; gx < 3; gx++) {
          const double vg = .125 * at_gauss(gx, r[0], r[1]), sg = vg * vg + eta;
          const bool comp = (cm >> ((gz * 3 + gy) * 3 + gx)) & 1u;
          s += gW(gx) * gW(gy) * gW(gz) * (comp ? (kap1 * (1. + eta) + 4. * mu1 * sg / 3.) * pw : sg);
        }
      }
  } else {
#pragma unroll
    for (int i = 7; i >= 0; i--) {
      const int o = __builtin_popcount(i);
      s += (o == 0 ? 1. : o == 1 ? 1. / 3. : o == 2 ? 1. / 9. : 1. / 27.) / 64. * (m[i] * m[i]);
    }
    s += eta;
  }
  out[e] = (E_elem ? E_elem[e] : E) * s;
}

// Coarse coefficients: the mean of the fine elements under a coarse one, by
// overlap.  Along one axis the fine elements lo .. lo + M - 1 meet coarse element
// C (nf / nc <= 2: at most three, two where the grids are nested or equal), with
// integer overlaps in units of 1 / nc that sum to nf (0 off the axis).
template <int M>
__device__ __forceinline__ void mg_overlap(int C, int nf, int nc, int (&e)[M], double (&w)[M]) {
  const int lo = mg_floor(C, nf, nc);
#pragma unroll
  for (int q = 0; q < M; q++) {
    const int d = mg_diff(lo + q, nc, C, nf);  // start of the fine element in the coarse one
    const int a = d > 0 ? d : 0, b = d + nc < nf ? d + nc : nf;
    w[q] = b > a && lo + q < nf ? (double)(b - a) : 0.;
    e[q] = lo + q < nf ? lo + q : nf - 1;
  }
}
template <int M>
__global__ __launch_bounds__(256) void k_mg_coarsen(Grid Gf, const double *__restrict__ cf, Grid Gc,
                                                    double *__restrict__ cc) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= (int64_t)Gc.nex * Gc.ney * Gc.nez) return;
  const int ci = (int)(c % Gc.nex), cj = (int)((c / Gc.nex) % Gc.ney), ck = (int)(c / ((int64_t)Gc.nex * Gc.ney));
  int x[M], y[M], z[M];
  double wx[M], wy[M], wz[M];
  mg_overlap<M>(ci, Gf.nex, Gc.nex, x, wx);
  mg_overlap<M>(cj, Gf.ney, Gc.ney, y, wy);
  mg_overlap<M>(ck, Gf.nez, Gc.nez, z, wz);
  double acc = 0.;
#pragma unroll
  for (int k = 0; k < M; k++)
#pragma unroll
    for (int j = 0; j < M; j++) {
      const double w = wy[j] * wz[k];
#pragma unroll
      for (int i = 0; i < M; i++) acc += (wx[i] * w) * cf[cell_id(Gf, x[i], y[j], z[k])];
    }
  cc[c] = acc / ((double)Gf.nex * Gf.ney * Gf.nez);
}
// FP32 inverse diagonal of a coarse level (s = 1): every element corner has
// E vol / 9 [(lam + mu) / h_c^2 + mu sum_d 1 / h_d^2] = E kc; 1 on the Dirichlet
// rows.  With the coefficients of its level about 8 us per level of a 32^3
// problem, 21 us with the marching diagonal kernel and a reciprocal pass.
__global__ __launch_bounds__(256) void k_mg_diag32(Grid G, const double *__restrict__ E, BcMask bc, double kx, double ky,
                                                   double kz, float *__restrict__ dinv) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (int64_t)G.nx * G.ny * G.nz) return;
  const int i = (int)(n % G.nx), j = (int)((n / G.nx) % G.ny), k = (int)(n / ((int64_t)G.nx * G.ny));
  double s = 0.;
#pragma unroll
  for (int a = 0; a < 8; a++) {
    const int ei = i - (a & 1), ej = j - ((a >> 1) & 1), ek = k - (a >> 2);
    if (ei >= 0 && ei < G.nex && ej >= 0 && ej < G.ney && ek >= 0 && ek < G.nez) s += E[cell_id(G, ei, ej, ek)];
  }
  const double kc[3] = {kx, ky, kz};
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const double d = kc[c] * s;
    dinv[3 * n + c] = on_dirichlet(G, bc.face[c], bc.vert[c], i, j, k) || d == 0. ? 1.f : (float)(1. / d);
  }
}

constexpr int PLANE_ROWS = 1 << 15;
__device__ __forceinline__ int plane_of_block() { return (int)(blockIdx.y + gridDim.y * blockIdx.z); }
static dim3 plane_grid(unsigned x, int nz) {
  return dim3(x, nz < PLANE_ROWS ? nz : PLANE_ROWS, (nz + PLANE_ROWS - 1) / PLANE_ROWS);
}

// Transfers, one plane of nodes per block row (so that indices are 32-bit; after
// PLANE_ROWS rows, under a launch's limit of 65535, they go on in z): restriction
// one thread per (coarse node, component), on small levels (latency-bound) four,
// one per fine plane of the gather; prolongation one thread per fine node.
// Restriction, mean of the 129^3 -> 65^3 -> 33^3 nodes 9.7 us (25 us as three
// separable passes that formed b - A x and the Dirichlet tests themselves), of
// 33^3 -> 17^3 -> 9^3 3.2 us (8.8 us with FP64 weights); prolongation, mean of
// the four levels of 128^3 8.0 us (9.8).
template <int M, int LANES>
__global__ __launch_bounds__(256) void k_mg_restrict(Grid Gf, Grid Gc, BcMask bc, const float *__restrict__ r,
                                                     float *__restrict__ bcoarse) {
  const int g = blockIdx.x * 256 + threadIdx.x, t = g / LANES, np = 3 * Gc.nx * Gc.ny;
  const int pl = plane_of_block(), K = pl < Gc.nz ? pl : 0;
  const bool ok = t < np && pl < Gc.nz;
  const int N = ok ? t / 3 : 0, c = ok ? t - 3 * N : 0, J = N / Gc.nx, I = N - J * Gc.nx;
  if constexpr (LANES == 1) {
    if (ok) bcoarse[t + (int64_t)np * K] = mg_restrict_entry<M>(Gf, Gc, bc, r, I, J, K, c);
  } else {
    const float v = mg_lanes(mg_restrict_plane<M>(Gf, Gc, bc, r, I, J, K, c, g & 3));
    if (ok && (g & 3) == 0) bcoarse[t + (int64_t)np * K] = v;
  }
}
template <bool NESTED>
__global__ __launch_bounds__(256) void k_mg_prolong(Grid Gf, Grid Gc, BcMask bc, const float *__restrict__ xc,
                                                    float *__restrict__ xf) {
  const int t = blockIdx.x * 256 + threadIdx.x, k = plane_of_block();
  if (t >= Gf.nx * Gf.ny || k >= Gf.nz) return;
  const int j = t / Gf.nx;
  mg_prolong_node<NESTED>(Gf, Gc, bc, xc, xf, t - j * Gf.nx, j, k);
}
// ----------------------------------------------------------------- smoother
__global__ void k_mg_cheb(const float *__restrict__ b, const float *__restrict__ y, const float *__restrict__ dinv,
                          float *__restrict__ d, float *__restrict__ x, float c1, float c2, int dfirst, int xzero,
                          int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) mg_cheb_entry(b, y, dinv, d, x, c1, c2, dfirst, xzero, i);
}

__global__ void k_mg_fill32(float *x, float v, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = v;
}

static unsigned nbm(int64_t n) { return (unsigned)((n + 255) / 256); }

void launch_mg_elem_coef(const DevProblem &P, double *out, hipStream_t s) {
  auto go = [&](auto k) {
    hipLaunchKernelGGL(k, dim3(nbm(P.ne)), dim3(256), 0, s, P.G, (const double *)P.V, (const double *)P.E_elem, P.E, P.eta,
                       (const uint32_t *)P.cmask, P.lam1, P.mu1, out);
  };
  P.unilateral ? go(k_mg_elem_coef<true>) : go(k_mg_elem_coef<false>);
}
void launch_mg_coarsen(const Grid &Gf, const double *cf, const Grid &Gc, double *cc, hipStream_t s) {
  const int64_t ne = (int64_t)Gc.nex * Gc.ney * Gc.nez;
  auto two = [](int f, int c) { return f == c || f == 2 * c; };
  auto go = [&](auto k) { hipLaunchKernelGGL(k, dim3(nbm(ne)), dim3(256), 0, s, Gf, cf, Gc, cc); };
  two(Gf.nex, Gc.nex) && two(Gf.ney, Gc.ney) && two(Gf.nez, Gc.nez) ? go(k_mg_coarsen<2>) : go(k_mg_coarsen<3>);
}
void launch_mg_restrict(const Grid &Gf, const Grid &Gc, const BcMask &bc, const float *r, float *bcoarse,
                        hipStream_t s) {
  const int64_t np = 3 * (int64_t)Gc.nx * Gc.ny;
  const bool small = np * Gc.nz <= (1 << 16);  // few entries: split each over its fine planes
  const dim3 g = plane_grid(nbm(small ? 4 * np : np), Gc.nz);
  auto go = [&](auto k) { hipLaunchKernelGGL(k, g, dim3(256), 0, s, Gf, Gc, bc, r, bcoarse); };
  if (mg_nested_grids(Gf, Gc)) small ? go(k_mg_restrict<3, 4>) : go(k_mg_restrict<3, 1>);
  else small ? go(k_mg_restrict<4, 4>) : go(k_mg_restrict<4, 1>);
}
void launch_mg_prolong(const Grid &Gf, const Grid &Gc, const BcMask &bc, const float *xc, float *xf,
                       hipStream_t s) {
  const dim3 g = plane_grid(nbm((int64_t)Gf.nx * Gf.ny), Gf.nz);
  if (mg_nested_grids(Gf, Gc)) hipLaunchKernelGGL(k_mg_prolong<true>, g, dim3(256), 0, s, Gf, Gc, bc, xc, xf);
  else hipLaunchKernelGGL(k_mg_prolong<false>, g, dim3(256), 0, s, Gf, Gc, bc, xc, xf);
}
void launch_mg_cheb(const float *b, const float *y, const float *dinv, float *d, float *x, float c1, float c2,
                    int dfirst, int xzero, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_mg_cheb, dim3(nbm(n)), dim3(256), 0, s, b, y, dinv, d, x, c1, c2, dfirst, xzero, n);
}
void launch_mg_diag32(const DevProblem &P, float *dinv, hipStream_t s) {
  const Grid &G = P.G;
  const double vol = G.hx * G.hy * G.hz / 9., i2[3] = {1. / (G.hx * G.hx), 1. / (G.hy * G.hy), 1. / (G.hz * G.hz)};
  double kc[3];
  for (int c = 0; c < 3; c++) kc[c] = vol * ((P.lam1 + P.mu1) * i2[c] + P.mu1 * (i2[0] + i2[1] + i2[2]));
  hipLaunchKernelGGL(k_mg_diag32, dim3(nbm(P.nn)), dim3(256), 0, s, G, (const double *)P.E_elem, P.bcU, kc[0], kc[1],
                     kc[2], dinv);
}
void launch_mg_fill32(float *x, float v, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_mg_fill32, dim3(nbm(n)), dim3(256), 0, s, x, v, n);
}
}  // namespace vfg
