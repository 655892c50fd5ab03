// vfg_internal.h -- device-side building blocks shared by the vfg kernels.
//
// Element basis: trilinear Q1 on an axis-aligned box, 3-point Gauss-Legendre
// per direction (27 points), exactly the rule of VFCartFEElement3DInit
// (VFCartFE.c:90-116, 216-269).  The 27-point tables are never stored: what
// visits the points does so by sum factorisation with the 1-D tables below, the
// rest works on polynomial moments (vfg_modal.h).
//
// Node accumulation ("gather") without atomics: a workgroup owns a tile of
// (TX-1) x (TY-1) node columns and marches upward through a z-chunk of node
// planes.  One thread computes one element of the (TX x TY) element columns
// that touch the owned nodes (a one-element halo is recomputed), element
// contributions are combined across the x neighbour with a lane shuffle and
// across the y neighbour through LDS, and the plane below the current element
// layer is complete after each step.  Every node sums its 8 element
// contributions in a fixed order, so results are bitwise reproducible.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include <utility>

namespace vfg {

// 1-D Gauss tables on [0,1]: P0[g] = phi_0(xi_g), P1[g] = phi_1(xi_g) and the
// weights w[g] (times the element length), VFCartFE.c:100-113.
#define VFG_SQ35 0.77459666924148337704  // sqrt(3/5)
__host__ __device__ constexpr double gP0(int g) { return g == 0 ? (1. + VFG_SQ35) * .5 : g == 1 ? .5 : (1. - VFG_SQ35) * .5; }
__host__ __device__ constexpr double gP1(int g) { return g == 0 ? (1. - VFG_SQ35) * .5 : g == 1 ? .5 : (1. + VFG_SQ35) * .5; }
__host__ __device__ constexpr double gW(int g) { return g == 1 ? 8. / 18. : 5. / 18.; }

struct Grid {
  int nx, ny, nz;     // nodes
  int nex, ney, nez;  // elements
  double hx, hy, hz;  // uniform element size
};

__device__ __forceinline__ int64_t node_id(const Grid &G, int i, int j, int k) {
  return (int64_t)i + (int64_t)G.nx * ((int64_t)j + (int64_t)G.ny * k);
}
__device__ __forceinline__ int64_t cell_id(const Grid &G, int i, int j, int k) {
  return (int64_t)i + (int64_t)G.nex * ((int64_t)j + (int64_t)G.ney * k);
}

// Workgroups go to the eight XCDs round-robin by linear id, and each XCD has
// its own L2.  xcd_block renumbers a 3-D grid so that XCD k runs one
// contiguous range of blocks in (x, y, z) order: tiles that are neighbours in
// x and y, whose halo node lines overlap, then meet in the same L2.
struct Blk3 {
  int x, y, z;
};
__device__ __forceinline__ Blk3 xcd_block() {
  const unsigned gx = gridDim.x, gy = gridDim.y, n = gx * gy * gridDim.z;
  const unsigned id = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
  const unsigned per = n / 8, rem = n % 8, x = id % 8, loc = id / 8;
  const unsigned l = (x < rem ? x * (per + 1) : rem * (per + 1) + (x - rem) * per) + loc;
  return Blk3{(int)(l % gx), (int)((l / gx) % gy), (int)(l / (gx * gy))};
}

// tr(eps(u)) at Gauss point (gx, gy, gz) of an element from its 8 nodal
// displacements (local node a = (k*2+j)*2+i), accumulated per component over
// the nodes and summed as (d1u1 + d2u2) + d3u3: the u operator, its diagonal and
// its loads branch on the sign of this value (UNILATERAL_NOCOMPRESSION).
__device__ __forceinline__ double tr_eps_at(const double (&u)[8][3], int gx, int gy, int gz, double ihx,
                                            double ihy, double ihz) {
  double h0 = 0., h1 = 0., h2 = 0.;
  for (int a = 0; a < 8; a++) {
    const int i = a & 1, j = (a >> 1) & 1, k = a >> 2;
    const double px = i ? gP1(gx) : gP0(gx), py = j ? gP1(gy) : gP0(gy), pz = k ? gP1(gz) : gP0(gz);
    h0 += (i ? ihx : -ihx) * py * pz * u[a][0];
    h1 += (j ? ihy : -ihy) * px * pz * u[a][1];
    h2 += (k ? ihz : -ihz) * px * py * u[a][2];
  }
  return (h0 + h1) + h2;
}
// bit g = (gz*3+gy)*3+gx set where tr(eps(u)) < 0 (UNILATERAL_THRES = 0, VFMech.c:6)
__device__ __forceinline__ uint32_t compression_mask(const double (&u)[8][3], double ihx, double ihy, double ihz) {
  uint32_t m = 0u;
  for (int g = 0; g < 27; g++)
    if (tr_eps_at(u, g % 3, (g / 3) % 3, g / 9, ihx, ihy, ihz) < 0.) m |= 1u << g;
  return m;
}

// Dirichlet row set of one component, computed from node indices
// (MatApplyDirichletBC, VFCartFE.c:1147-1296): bit f of `face` set iff face f
// is not NONE; bit v of `vert` set iff vertex v is not NONE.
struct BcMask {
  uint8_t face[3];
  uint8_t vert[3];
};

__device__ __forceinline__ bool on_dirichlet(const Grid &G, uint8_t face, uint8_t vert, int i, int j,
                                             int k) {
  bool m = ((face & 1) && i == 0) || ((face & 2) && i == G.nx - 1) || ((face & 4) && j == 0) ||
           ((face & 8) && j == G.ny - 1) || ((face & 16) && k == 0) || ((face & 32) && k == G.nz - 1);
  if (vert) {
    int ix = (i == 0) ? 0 : (i == G.nx - 1) ? 1 : -1;
    int iy = (j == 0) ? 0 : (j == G.ny - 1) ? 1 : -1;
    int iz = (k == 0) ? 0 : (k == G.nz - 1) ? 1 : -1;
    if (ix >= 0 && iy >= 0 && iz >= 0 && ((vert >> (ix + 2 * iy + 4 * iz)) & 1)) m = true;
  }
  return m;
}

// wave64 / block reductions in FP64 with a fixed order (deterministic)
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
template <int NT>
__device__ __forceinline__ double block_sum(double v, double *sh /* NT/64 */) {
  v = wave_sum(v);
  const int w = threadIdx.x / 64, l = threadIdx.x % 64;
  if (l == 0) sh[w] = v;
  __syncthreads();
  double s = 0.;
  if (threadIdx.x == 0)
    for (int i = 0; i < NT / 64; i++) s += sh[i];
  __syncthreads();
  return s;  // valid in thread 0
}

// Vector chunks: the entries k = tid + u B of [0, len), four of a thread in
// flight at once (load(k), then work(k, value) in order).  Past the end a thread
// loads its first entry again: no other thread writes that.
template <int B, class L, class W>
__device__ __forceinline__ void chunk_walk(int len, const L &load, const W &work) {
  using R = decltype(load(0));
  for (int k0 = threadIdx.x; k0 < len; k0 += 4 * B) {
    R v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) v[u] = load(k0 + u * B < len ? k0 + u * B : k0);
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (k0 + u * B < len) work(k0 + u * B, v[u]);
  }
}
// entries per chunk of a member's vectors of n entries (a rule on the member
// alone: its partial sums do not depend on the others).  1024 = one round of
// loads in flight per workgroup of 256; the update of x and r in an engine of 8
// requests took 14.7 us in chunks of 4096, one entry in flight, and 5.2 us so.
// Long vectors fill the device either way, and each chunk is a partial to sum:
// batched u-solve of one cube in chunks of 1024 and 4096, 33^3 nodes 1.51 and 1.58
// ms, 65^3 2.42 and 2.43, 89^3 (2.1 M entries) 3.47 and 3.46, 97^3 3.96 and 3.91,
// 113^3 5.15 and 5.03.
inline int chunk_entries(int64_t n) { return n <= (1 << 21) ? 1024 : 4096; }

// ---------------------------------------------------------------- marching
// Op interface:
//   static constexpr int NF  -- staged nodal scalar fields
//   static constexpr int NC  -- accumulated components per node
//   __device__ T load(int f, int64_t node)  -- value of staged field f at a node
//   __device__ void element(int ex,int ey,int ek, const T (&xin)[2][4][NF], T (&r)[8][NC])
//   __device__ void store(int i,int j,int k, const T (&acc)[NC], const T (&own)[NF])
// Optional per-element coefficients read one layer ahead (hides their latency):
//   __device__ A aux(int ex,int ey,int ek); element(ex,ey,ek, xin, aux, r)
// with A any trivially copyable type (a value, or a struct of values).
// Corners of an element are a = (k*2+j)*2+i; xin[k][j*2+i][f].
template <class Op, class = void>
struct has_aux : std::false_type {};
template <class Op>
struct has_aux<Op, std::void_t<decltype(&Op::aux)>> : std::true_type {};
// Ops that also reduce over their owned nodes define
//   __device__ double store(...)      (returns the node's contribution)
//   __device__ void partial(int slot, double sum)
// the march sums the contributions of each thread, reduces them over the
// workgroup in a fixed order and hands the sum to partial(rslot, .).
template <class Op, class = void>
struct has_red : std::false_type {};
template <class Op>
struct has_red<Op, std::void_t<decltype(&Op::partial)>> : std::true_type {};

template <class Op, class = void>
struct aux_of {
  using type = int;
};
template <class Op>
struct aux_of<Op, std::void_t<decltype(&Op::aux)>> {
  using type = decltype(std::declval<const Op &>().aux(0, 0, 0));
};

template <typename T, int TX, int TY, class Op>
__device__ __forceinline__ void march(const Grid &G, const Op &op, int OZ, int bx, int by, int bz) {
  constexpr int NF = Op::NF, NC = Op::NC;
  constexpr int NT = TX * TY, OX = TX - 1, OY = TY - 1, SX = TX + 1, SY = TY + 1;
  constexpr int NPF = (SX * SY + NT - 1) / NT;  // staged nodes per thread
  constexpr bool AUX = has_aux<Op>::value;
  __shared__ T s_in[NF][SY * SX];
  __shared__ T s_red[2 * NC][NT];
  const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
  const int ox0 = bx * OX, oy0 = by * OY, oz0 = bz * OZ;
  const int ex = ox0 - 1 + tx, ey = oy0 - 1 + ty;
  const bool exy_ok = ex >= 0 && ex < G.nex && ey >= 0 && ey < G.ney;
  const bool owner = tx < OX && ty < OY && (ox0 + tx) < G.nx && (oy0 + ty) < G.ny;
  const int64_t plane = (int64_t)G.nx * G.ny;

  // staged nodes of this thread: in-plane offsets, fixed for the whole march
  int64_t soff[NPF];
  bool sok[NPF];
#pragma unroll
  for (int q = 0; q < NPF; q++) {
    const int n = tid + q * NT;
    const int lx = n % SX, ly = n / SX;
    const int gx = ox0 - 1 + lx, gy = oy0 - 1 + ly;
    sok[q] = n < SX * SY && gx >= 0 && gx < G.nx && gy >= 0 && gy < G.ny;
    soff[q] = sok[q] ? (int64_t)gx + (int64_t)G.nx * gy : 0;
  }
  // The next node plane is loaded into registers while the current element
  // layer computes, and written to LDS after the next barrier.
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
  auto commit = [&]() {
#pragma unroll
    for (int q = 0; q < NPF; q++) {
      const int n = tid + q * NT;
      if (n < SX * SY)
#pragma unroll
        for (int f = 0; f < NF; f++) s_in[f][n] = pf[q][f];
    }
  };
  using AuxT = typename aux_of<Op>::type;
  auto aux_at = [&](int ek) -> AuxT {
    AuxT a{};
    if constexpr (AUX) {
      if (exy_ok && ek >= 0 && ek < G.nez) a = op.aux(ex, ey, ek);
    }
    return a;
  };
  auto read_plane = [&](T (&xp)[4][NF]) {
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int f = 0; f < NF; f++) xp[q][f] = s_in[f][(ty + (q >> 1)) * SX + tx + (q & 1)];
  };
  T carry[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) carry[c] = T(0);
  // one element layer: bottom plane xb (node plane ek), top plane xt (ek + 1)
  auto layer = [&](int ek, const T (&xb)[4][NF], T (&xt)[4][NF], AuxT &aux_next) {
    const AuxT aux_cur = aux_next;
    __syncthreads();
    commit();       // plane ek + 1
    fetch(ek + 2);  // in flight during this layer
    aux_next = aux_at(ek + 1);
    __syncthreads();
    read_plane(xt);
    T r[8][NC];
#pragma unroll
    for (int a = 0; a < 8; a++)
#pragma unroll
      for (int c = 0; c < NC; c++) r[a][c] = T(0);
    if (exy_ok && ek >= 0 && ek < G.nez) {
      T xin[2][4][NF];
#pragma unroll
      for (int q = 0; q < 4; q++)
#pragma unroll
        for (int f = 0; f < NF; f++) {
          xin[0][q][f] = xb[q][f];
          xin[1][q][f] = xt[q][f];
        }
      if constexpr (AUX) op.element(ex, ey, ek, xin, aux_cur, r);
      else op.element(ex, ey, ek, xin, r);
    }
    // x-combine: node (ex+1) gets corner i=1 of this element and corner i=0
    // of the element to the right (next lane inside the 16-lane row).
    T cx[2][2][NC];
#pragma unroll
    for (int kz = 0; kz < 2; kz++)
#pragma unroll
      for (int jy = 0; jy < 2; jy++)
#pragma unroll
        for (int c = 0; c < NC; c++) {
          T right = __shfl_down(r[(kz * 2 + jy) * 2 + 0][c], 1, TX);
          cx[kz][jy][c] = r[(kz * 2 + jy) * 2 + 1][c] + right;
        }
    // y-combine through LDS: node (ey+1) gets row jy=1 of this element row and
    // row jy=0 of the element row above.
#pragma unroll
    for (int kz = 0; kz < 2; kz++)
#pragma unroll
      for (int c = 0; c < NC; c++) s_red[kz * NC + c][tid] = cx[kz][0][c];
    __syncthreads();
    if (owner) {
      T bot[NC];
#pragma unroll
      for (int c = 0; c < NC; c++) {
        bot[c] = carry[c] + (cx[0][1][c] + s_red[c][tid + TX]);
        carry[c] = cx[1][1][c] + s_red[NC + c][tid + TX];
      }
      if (ek >= oz0 && ek >= 0) op.store(ox0 + tx, oy0 + ty, ek, bot, xb[3]);
    }
  };

  T xa[4][NF], xb2[4][NF];  // ping-pong planes: no register copies between layers
  fetch(oz0 - 1);
  commit();
  fetch(oz0);
  AuxT aux_next = aux_at(oz0 - 1);
  __syncthreads();
  read_plane(xa);
  const int ek_end = min(oz0 + OZ - 1, G.nz - 1);
  for (int ek = oz0 - 1; ek <= ek_end; ek += 2) {
    layer(ek, xa, xb2, aux_next);
    if (ek + 1 > ek_end) break;
    layer(ek + 1, xb2, xa, aux_next);
  }
}

// march with the node planes kept in LDS.  Three planes rotate through LDS
// (bottom and top of the current element layer, and the one being committed
// for the next layer), so the element computation can re-read its corners
// instead of keeping them in registers:
//   __device__ void element_lds(int ex, int ey, int ek, const XS &xs, T (&r)[8][NC])
// with xs(k, q, f) the value of staged field f at corner (k, q = j*2+i).  The combination of
// the element results (x by lane shuffles, y through LDS, z carried) and the
// stores are those of march.  Two barriers per layer.  The next plane is loaded
// at the start of its layer; its latency is left to the other resident workgroup.
template <typename T, int TX, int TY, class Op>
__device__ __forceinline__ void march_lds(const Grid &G, const Op &op, int OZ, int bx, int by, int bz,
                                          int rslot = 0) {
  constexpr int NF = Op::NF, NC = Op::NC;
  constexpr int NT = TX * TY, OX = TX - 1, OY = TY - 1, SX = TX + 1, SY = TY + 1, PL = SX * SY;
  constexpr int NPF = (PL + NT - 1) / NT;
  constexpr bool RED = has_red<Op>::value;
  double racc = 0.;  // owned-node contributions (reducing ops)
  __shared__ T s_in[3][NF][PL];
  __shared__ T s_red[2 * NC][NT];
  const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
  const int ox0 = bx * OX, oy0 = by * OY, oz0 = bz * OZ;
  const int ex = ox0 - 1 + tx, ey = oy0 - 1 + ty;
  const bool exy_ok = ex >= 0 && ex < G.nex && ey >= 0 && ey < G.ney;
  const bool owner = tx < OX && ty < OY && (ox0 + tx) < G.nx && (oy0 + ty) < G.ny;
  const int64_t plane = (int64_t)G.nx * G.ny;
  int64_t soff[NPF];
  bool sok[NPF];
#pragma unroll
  for (int q = 0; q < NPF; q++) {
    const int n = tid + q * NT;
    const int lx = n % SX, ly = n / SX;
    const int gx = ox0 - 1 + lx, gy = oy0 - 1 + ly;
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
  const int c0 = ty * SX + tx;  // corner (j, i) = (0, 0) of this thread's element in a plane
  T carry[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) carry[c] = T(0);

  // planes rotate through the buffers: bottom bb, top bt, next bn
  int bb = 0, bt = 1, bn = 2;
  fetch(oz0 - 1);
  commit(bb);
  const int ek_end = min(oz0 + OZ - 1, G.nz - 1);
  for (int ek = oz0 - 1; ek <= ek_end; ek++) {
    // buffer bt last held a plane read two layers ago; the barriers since
    // then order this write after those reads
    fetch(ek + 1);
    commit(bt);
    __syncthreads();
    T r[8][NC];
#pragma unroll
    for (int a = 0; a < 8; a++)
#pragma unroll
      for (int c = 0; c < NC; c++) r[a][c] = T(0);
    if (exy_ok && ek >= 0 && ek < G.nez) {
      const T *pb = &s_in[bb][0][c0], *pt = &s_in[bt][0][c0];
      auto xs = [pb, pt](int k, int q, int f) -> T {
        return (k ? pt : pb)[f * PL + (q >> 1) * SX + (q & 1)];
      };
      op.element_lds(ex, ey, ek, xs, r);
    }
    T cx[2][2][NC];
#pragma unroll
    for (int kz = 0; kz < 2; kz++)
#pragma unroll
      for (int jy = 0; jy < 2; jy++)
#pragma unroll
        for (int c = 0; c < NC; c++) {
          T right = __shfl_down(r[(kz * 2 + jy) * 2 + 0][c], 1, TX);
          cx[kz][jy][c] = r[(kz * 2 + jy) * 2 + 1][c] + right;
        }
#pragma unroll
    for (int kz = 0; kz < 2; kz++)
#pragma unroll
      for (int c = 0; c < NC; c++) s_red[kz * NC + c][tid] = cx[kz][0][c];
    __syncthreads();
    if (owner) {
      T bot[NC], own[NF];
#pragma unroll
      for (int c = 0; c < NC; c++) {
        bot[c] = carry[c] + (cx[0][1][c] + s_red[c][tid + TX]);
        carry[c] = cx[1][1][c] + s_red[NC + c][tid + TX];
      }
      if (ek >= oz0 && ek >= 0) {
#pragma unroll
        for (int f = 0; f < NF; f++) own[f] = s_in[bb][f][c0 + SX + 1];
        if constexpr (RED) racc += op.store(ox0 + tx, oy0 + ty, ek, bot, own);
        else op.store(ox0 + tx, oy0 + ty, ek, bot, own);
      }
    }
    const int b = bb;
    bb = bt;
    bt = bn;
    bn = b;
  }
  if constexpr (RED) {
    __shared__ double s_rs[NT / 64];
    const double v = block_sum<NT>(racc, s_rs);
    if (tid == 0) op.partial(rslot, v);
  }
}

template <typename T>
__device__ __forceinline__ T interp(int g, T f0, T f1) {
  return T(gP0(g)) * f0 + T(gP1(g)) * f1;
}

// the march at a renumbered block (xcd_block)
template <typename T, int TX, int TY, class Op>
__device__ __forceinline__ void march(const Grid &G, const Op &op, int OZ, Blk3 b) {
  march<T, TX, TY>(G, op, OZ, b.x, b.y, b.z);
}

}  // namespace vfg
