// vfg_mg.h -- grid-transfer device code shared by the single-problem and the
// batched multigrid (internal).
#pragma once
#include "vfg_internal.h"

namespace vfg {

// Coarse grids cover the same box with ceil(n/2) elements per direction
// (directions already at the minimum keep theirs), so the grids are nested
// only where n is even.  Everything between two levels is built from the 1-D
// map xi(i) = i * nc / nf of fine node i onto the coarse node axis:
//   prolongation: trilinear interpolation at xi, weight 1 - |xi - I| for the
//     two coarse nodes I bracketing xi;
//   restriction: its transpose (the same weights, gathered per coarse node);
//   coefficients: the overlap-weighted mean of the fine elements under each
//     coarse element.
// The weights are formed from integers, (nf - |i nc - I nf|) / nf, and written
// out (1/2, 1, 1/2) where the grids are nested.  A product of two counts passes
// 31 bits on an axis of more than 65535 elements, so quotients are written out
// for the pairs in use (nc = nf or ceil(nf / 2)) and differences of products,
// which are a few nf at most, are formed modulo 2^32.
// floor(C nf / nc), 0 <= C < nc
__device__ __forceinline__ int mg_floor(int C, int nf, int nc) {
  return nf == nc ? C : 2 * C - (nf < 2 * nc && C > 0 ? 1 : 0);
}
// i nc - I nf
__device__ __forceinline__ int mg_diff(int i, int nc, int I, int nf) {
  return (int)((unsigned)i * (unsigned)nc - (unsigned)I * (unsigned)nf);
}
__host__ __device__ __forceinline__ bool mg_nested_grids(const Grid &Gf, const Grid &Gc) {
  return Gf.nex == 2 * Gc.nex && Gf.ney == 2 * Gc.ney && Gf.nez == 2 * Gc.nez;
}

// ------------------------------------------------- restriction / prolongation
// both transfers take their weights from here, so they are each other's transpose
__device__ __forceinline__ float mg_wt(int n, int nf) { return (float)n / (float)nf; }
// The fine nodes i0 .. i0 + M - 1 of one axis that coarse node I gathers from,
// with weights, zero off the axis and outside the hat (i is clamped to the
// axis, so every load is in range).  M = 3: nested; 4: nf / nc <= 2.
template <int M>
__device__ __forceinline__ void mg_gather(int I, int nf, int nc, int (&i)[M], float (&w)[M]) {
  if constexpr (M == 3) {
#pragma unroll
    for (int q = 0; q < 3; q++) {
      i[q] = 2 * I - 1 + q;
      w[q] = i[q] < 0 || i[q] > nf ? 0.f : q == 1 ? 1.f : .5f;
    }
  } else {
    const int lo = I > 0 ? mg_floor(I - 1, nf, nc) + 1 : 0;  // first i with i nc > (I - 1) nf
#pragma unroll
    for (int q = 0; q < M; q++) {
      i[q] = lo + q;
      const int m = mg_diff(i[q], nc, I, nf), n = nf - (m < 0 ? -m : m);
      w[q] = n <= 0 || i[q] > nf ? 0.f : mg_wt(n, nf);
    }
  }
#pragma unroll
  for (int q = 0; q < M; q++) i[q] = i[q] < 0 ? 0 : i[q] > nf ? nf : i[q];
}

// Lane kk (< 4) of coarse rhs entry (node (I, J, K), component c) = P^T r, r
// zero on the fine Dirichlet rows: fine plane kk of the gather.  The entry is
// the sum over the four lanes (mg_lanes), 0 on the coarse Dirichlet rows.  All
// M^2 loads of a lane are independent of each other.
template <int M>
__device__ __forceinline__ float mg_restrict_plane(const Grid &Gf, const Grid &Gc, const BcMask &bc,
                                                   const float *__restrict__ r, int I, int J, int K, int c, int kk) {
  if (on_dirichlet(Gc, bc.face[c], bc.vert[c], I, J, K)) return 0.f;
  int i[M], j[M], k[M];
  float wx[M], wy[M], wz[M];
  mg_gather<M>(I, Gf.nex, Gc.nex, i, wx);
  mg_gather<M>(J, Gf.ney, Gc.ney, j, wy);
  mg_gather<M>(K, Gf.nez, Gc.nez, k, wz);
  int kp = 0;
  float wp = 0.f;
#pragma unroll
  for (int q = 0; q < M; q++)
    if (q == kk) {
      kp = k[q];
      wp = wz[q];
    }
  float pl = 0.f;
#pragma unroll
  for (int jj = 0; jj < M; jj++) {
    const float *__restrict__ row = r + 3 * ((int64_t)Gf.nx * (j[jj] + (int64_t)Gf.ny * kp)) + c;
    float s = 0.f;
#pragma unroll
    for (int ii = 0; ii < M; ii++) s += wx[ii] * row[3 * i[ii]];
    pl += wy[jj] * s;
  }
  return wp * pl;
}
// one thread per entry: the same value (planes summed in lane order)
template <int M>
__device__ __forceinline__ float mg_restrict_entry(const Grid &Gf, const Grid &Gc, const BcMask &bc,
                                                   const float *__restrict__ r, int I, int J, int K, int c) {
  float v = 0.f;
#pragma unroll
  for (int kk = 0; kk < M; kk++) v += mg_restrict_plane<M>(Gf, Gc, bc, r, I, J, K, c, kk);
  return v;
}
// sum over four lanes in lane order, in the first of them
__device__ __forceinline__ float mg_lanes(float v) {
  const float v1 = __shfl_down(v, 1, 4), v2 = __shfl_down(v, 2, 4), v3 = __shfl_down(v, 3, 4);
  return ((v + v1) + v2) + v3;
}

// the two coarse nodes around fine node i of one axis, with weights (the second
// is the first again where its weight is 0)
template <bool NESTED>
__device__ __forceinline__ void mg_bracket(int i, int nf, int nc, int (&I)[2], float (&w)[2]) {
  if constexpr (NESTED) {
    I[0] = i >> 1;
    I[1] = I[0] + (i & 1);
    w[0] = i & 1 ? .5f : 1.f;
    w[1] = i & 1 ? .5f : 0.f;
  } else {
    const int q = nf == nc ? i : i == nf ? nc : i >> 1, m = mg_diff(i, nc, q, nf);
    I[0] = q;
    I[1] = q + (m > 0);
    w[0] = mg_wt(nf - m, nf);
    w[1] = mg_wt(m, nf);
  }
}
// x_fine(node (i, j, k)) += P x_coarse on the free fine rows
template <bool NESTED>
__device__ __forceinline__ void mg_prolong_node(const Grid &Gf, const Grid &Gc, const BcMask &bc,
                                                const float *__restrict__ xc, float *__restrict__ xf, int i, int j,
                                                int k) {
  int I[2], J[2], K[2];
  float wx[2], wy[2], wz[2];
  mg_bracket<NESTED>(i, Gf.nex, Gc.nex, I, wx);
  mg_bracket<NESTED>(j, Gf.ney, Gc.ney, J, wy);
  mg_bracket<NESTED>(k, Gf.nez, Gc.nez, K, wz);
  float *__restrict__ p = xf + 3 * node_id(Gf, i, j, k);
  float x[3], acc[3] = {0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < 3; c++) x[c] = p[c];
#pragma unroll
  for (int c3 = 0; c3 < 2; c3++)
#pragma unroll
    for (int c2 = 0; c2 < 2; c2++) {
      const float *__restrict__ row = xc + 3 * ((int64_t)Gc.nx * (J[c2] + (int64_t)Gc.ny * K[c3]));
      const float w = wz[c3] * wy[c2];
#pragma unroll
      for (int c = 0; c < 3; c++) acc[c] += w * (wx[0] * row[3 * I[0] + c] + wx[1] * row[3 * I[1] + c]);
    }
#pragma unroll
  for (int c = 0; c < 3; c++)
    if (!on_dirichlet(Gf, bc.face[c], bc.vert[c], i, j, k)) p[c] = x[c] + acc[c];
}

// one Chebyshev step on the Jacobi-scaled system, entry i:
//   res = b - y (use_y) or b;  d = c1 d + c2 D^-1 res (dfirst: c2 D^-1 res);
//   x = x + d (xzero: x = d)
__device__ __forceinline__ void mg_cheb_entry(const float *__restrict__ b, const float *__restrict__ y,
                                              const float *__restrict__ dinv, float *__restrict__ d,
                                              float *__restrict__ x, float c1, float c2, int dfirst, int xzero,
                                              int64_t i) {
  const float res = y ? b[i] - y[i] : b[i];
  const float di = (dfirst ? 0.f : c1 * d[i]) + c2 * dinv[i] * res;
  d[i] = di;
  x[i] = xzero ? di : x[i] + di;
}

}  // namespace vfg
