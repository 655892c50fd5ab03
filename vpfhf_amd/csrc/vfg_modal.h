// vfg_modal.h -- the z-march of the operators whose element is a polynomial
// (moment) form; see vfg_umodal.h for the elasticity element and vfg_v.hip for
// the phase-field one.
//
// Notation: on an element (xi, eta, zeta in [-1,1]) a nodal field is
// sum F_abc xi^a eta^b zeta^c / 8 with F_abc the signed sums of its corner
// values; the modal sums of one face (node plane) are F_ab = s, x, y, w for
// ab = 00, 10, 01, 11.  Dually the forces at the corners are the signed sums of
// eight modal forces.
#pragma once
#include "vfg_internal.h"

namespace vfg {

// modal index i = a + 2 b + 4 c of xi^a eta^b zeta^c: power of variable d
constexpr int um_pow(int i, int d) { return (i >> d) & 1; }

// the modal sums of the corner values cv(a), derivatives from nodal differences
template <typename CV>
__device__ __forceinline__ void modal_sums(const CV &cv, double (&m)[8]) {
  double f[2][5];  // per face: first corner, and of the differences to it the sum, x, y, twist
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const double x0 = cv(k * 4), b = cv(k * 4 + 1) - x0, e = cv(k * 4 + 2) - x0, d = cv(k * 4 + 3) - x0, t = d - e;
    f[k][0] = x0;
    f[k][2] = t + b;
    f[k][4] = t - b;
    f[k][3] = 2. * d - f[k][2];
    f[k][1] = 2. * d - f[k][4];
  }
  m[0] = 4. * (f[0][0] + f[1][0]) + (f[0][1] + f[1][1]);
  m[4] = 4. * (f[1][0] - f[0][0]) + (f[1][1] - f[0][1]);
#pragma unroll
  for (int q = 1; q < 4; q++) {
    m[q] = f[1][q + 1] + f[0][q + 1];
    m[q + 4] = f[1][q + 1] - f[0][q + 1];
  }
}
// modal index with power t of variable d and powers b, c of the two others
constexpr int modal_at(int d, int t, int b, int c) {
  const int o1 = d == 0 ? 1 : 0, o2 = d == 2 ? 1 : 2;
  return t << d | b << o1 | c << o2;
}
constexpr double gX(int g) { return (g - 1) * VFG_SQ35; }  // Gauss point of [-1, 1]
// a + b x at Gauss point g
__device__ __forceinline__ double at_gauss(int g, double a, double b) { return g == 1 ? a : a + gX(g) * b; }
// the averages of P D x^a y^b over the square, a, b <= 1, of two bilinear
// functions given by their coefficients, each still to be divided by 3^(a + b)
__device__ __forceinline__ void bilinear_moments(const double (&P)[2][2], const double (&D)[2][2], double (&M)[2][2]) {
  double c[2][2][2];  // [power of x][power of y in P][in D]
#pragma unroll
  for (int b = 0; b < 2; b++)
#pragma unroll
    for (int e = 0; e < 2; e++) {
      c[0][b][e] = P[0][b] * D[0][e] + (1. / 3.) * (P[1][b] * D[1][e]);
      c[1][b][e] = P[0][b] * D[1][e] + P[1][b] * D[0][e];
    }
#pragma unroll
  for (int a = 0; a < 2; a++) {
    M[a][0] = c[a][0][0] + (1. / 3.) * c[a][1][1];
    M[a][1] = c[a][0][1] + c[a][1][0];
  }
}

// tile-blocked coefficients: [tile][element layer][wavefront][coefficient][64
// slots]; a wavefront reads and writes each coefficient as one aligned 512-byte
// segment and all of them as one block.  Halo elements are stored in every tile
// that computes them.  (V set-up and apply are 1 % faster than with each
// coefficient's segments of the four wavefronts together.)
__host__ __device__ inline int64_t tiled_index(int tile, int ek, int nez, int ncoef, int slot) {
  return (((int64_t)tile * nez + ek) * 4 + slot / 64) * ncoef * 64 + slot % 64;
}

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
// the vertex (VFG_X0Y0Z0..) of a node that lies on three faces, else -1
__device__ __forceinline__ int face_vertex(uint32_t fb) {
  if (!((fb & 3u) && (fb & 12u) && (fb & 48u))) return -1;
  return (int)((fb >> 1 & 1u) + 2u * (fb >> 3 & 1u) + 4u * (fb >> 5 & 1u));
}
// on_dirichlet from the face bits
__device__ __forceinline__ bool face_dirichlet(uint8_t face, uint8_t vert, uint32_t fb) {
  bool m = (face & fb) != 0u;
  if (vert) {
    const int v = face_vertex(fb);
    if (v >= 0) m = m || ((vert >> v) & 1);
  }
  return m;
}

// A workgroup owns (TX-1) x (TY-1) node columns, computes the TX x TY element
// columns that touch them (a one-element halo is recomputed) and marches up a
// z-chunk of OZ node planes.  Every node sums its eight element contributions
// in a fixed order.
//   - A thread keeps what it needs of the two node planes of its element
//     (Op::Face), not the corners, and the plane under construction as four
//     modal sums per component: an element adds its bottom part to the carried
//     plane, and only that one plane is turned into nodal values and combined
//     with the x and y neighbours per layer (lane shift along x, LDS along y).
//   - The y-combination and the store of a plane happen after the next
//     layer's barrier, so a layer has one barrier (s_in and s_red alternate
//     between two buffers: a buffer is written again two barriers after its
//     last read).
//   - The next plane and the element's coefficients are loaded a layer ahead;
//     the first two planes are loaded together.
// Op interface:
//   T, NF, NC, Face, Aux, Own         value type, staged fields, components, types
//   Raw load(f, n); T stage(f, raw)   staged field f at node n: what is loaded a layer
//                                     ahead, and its value, formed when it is needed (an
//                                     operation on a load at once would wait for it)
//   Raw off()                         (static) what stages to 0: nodes off the grid
//   face(rd, F)                       F from the corner values rd(f, q), q = 2 j + i
//   Own own(F)                        what store needs of the thread's own node (q = 3)
//   Aux aux(ex, ey, ek, tile, slot)   the element's coefficients
//   element(a, B, F, tot, carry)      adds the modal forces of the layer between
//                                     faces B and F: the bottom ones to tot, sets
//                                     the top ones in carry
//   O own_load(n)                     (optional) data of an owned node, read a layer before its store
//   store(n, fb, acc, own[, o])       fb: face bits of the node
//   partial(slot, sum)                (optional) the workgroup's sum of what store returned
template <class Op, class = void>
struct has_own : std::false_type {};
template <class Op>
struct has_own<Op, std::void_t<decltype(&Op::own_load)>> : std::true_type {};
template <class Op, class = void>
struct ownm_of {
  using type = int;
};
template <class Op>
struct ownm_of<Op, std::void_t<decltype(&Op::own_load)>> {
  using type = decltype(std::declval<const Op &>().own_load(int64_t(0)));
};

template <int TX, int TY, class Op>
__device__ __forceinline__ void march_modal(const Grid &G, const Op &op, int OZ, int bx, int by, int bz,
                                            int rslot = 0) {
  static_assert(TX == 8 || TX == 16, "the x-combination shifts inside 16-lane rows");
  using T = typename Op::T;
  constexpr int NF = Op::NF, NC = Op::NC;
  constexpr int NT = TX * TY, OX = TX - 1, OY = TY - 1, SX = TX + 1, PL = SX * (TY + 1);
  constexpr int NPF = (PL + NT - 1) / NT;
  constexpr bool RED = has_red<Op>::value, OWN = has_own<Op>::value;
  __shared__ T s_in[2][NF][PL];
  __shared__ T s_red[2][NC][NT];
  const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
  const int ox0 = bx * OX, oy0 = by * OY, oz0 = bz * OZ;
  const int ex = ox0 - 1 + tx, ey = oy0 - 1 + ty;
  const bool exy_ok = ex >= 0 && ex < G.nex && ey >= 0 && ey < G.ney;
  const bool owner = tx < OX && ty < OY && (ox0 + tx) < G.nx && (oy0 + ty) < G.ny;
  const int64_t plane = (int64_t)G.nx * G.ny;
  const uint32_t fbxy = face_bits_xy(G, ox0 + tx, oy0 + ty);
  const int tile = bx + ((G.nx + OX - 1) / OX) * by;
  const int ek0 = oz0 - 1, ek_end = min(oz0 + OZ - 1, G.nz - 1);
  int64_t nst = (int64_t)(ox0 + tx) + (int64_t)G.nx * (oy0 + ty) + plane * ek0;  // owned node of the plane stored next

  int64_t soff[NPF];  // staged nodes of this thread in the plane fetched next
  bool sok[NPF];
#pragma unroll
  for (int q = 0; q < NPF; q++) {
    const int n = tid + q * NT;
    const int gx = ox0 - 1 + n % SX, gy = oy0 - 1 + n / SX;
    sok[q] = n < PL && gx >= 0 && gx < G.nx && gy >= 0 && gy < G.ny;
    soff[q] = (sok[q] ? (int64_t)gx + (int64_t)G.nx * gy : 0) + plane * ek0;
  }
  using Raw = typename Op::Raw;
  Raw pf[NPF][NF];
  auto fetch = [&](int iz, Raw (&v)[NPF][NF]) {
    const bool zok = iz >= 0 && iz < G.nz;  // uniform
#pragma unroll
    for (int q = 0; q < NPF; q++) {
      const bool ok = zok && sok[q];
#pragma unroll
      for (int f = 0; f < NF; f++) {
        if (ok) v[q][f] = op.load(f, soff[q]);
        else v[q][f] = Op::off();
      }
      soff[q] += plane;
    }
  };
  auto commit = [&](int b, const Raw (&v)[NPF][NF]) {
#pragma unroll
    for (int q = 0; q < NPF; q++) {
      const int n = tid + q * NT;
      if (n < PL)
#pragma unroll
        for (int f = 0; f < NF; f++) s_in[b][f][n] = op.stage(f, v[q][f]);
    }
  };
  const int c0 = ty * SX + tx;
  using Face = typename Op::Face;
  auto read_face = [&](int b, Face &F) {
    op.face([&](int f, int q) -> T { return s_in[b][f][c0 + (q >> 1) * SX + (q & 1)]; }, F);
  };
  using Aux = typename Op::Aux;
  // off the grid the coefficients stay as they are: they are not used there
  auto aux_at = [&](int ek, Aux &a) {
    if (exy_ok && ek >= 0 && ek < G.nez) a = op.aux(ex, ey, ek, tile, tid);
  };
  using OwnT = typename ownm_of<Op>::type;

  T carry[NC][4];  // modal sums of the node plane on top of the last layer
#pragma unroll
  for (int c = 0; c < NC; c++)
#pragma unroll
    for (int q = 0; q < 4; q++) carry[c][q] = T(0);
  T pend[NC] = {};  // this thread's part of the plane waiting for its y-combination
  typename Op::Own pown{};
  OwnT po{};
  double racc = 0.;
  auto finish = [&](int k, int b) {
    if (owner && k >= oz0) {
      T acc[NC];
#pragma unroll
      for (int c = 0; c < NC; c++) acc[c] = pend[c] + s_red[b][c][tid + TX];
      const uint32_t fb = fbxy | (k == 0 ? 16u : 0u) | (k == G.nz - 1 ? 32u : 0u);
      if constexpr (OWN) {
        if constexpr (RED) racc += op.store(nst, fb, acc, pown, po);
        else op.store(nst, fb, acc, pown, po);
      } else {
        if constexpr (RED) racc += op.store(nst, fb, acc, pown);
        else op.store(nst, fb, acc, pown);
      }
    }
    nst += plane;
  };
  // one element layer between node planes ek (B) and ek + 1 (F)
  auto layer = [&](int ek, const Face &B, Face &F, Aux &a_next) {
    const Aux a = a_next;
    const int b = (ek - ek0) & 1;
    commit(b ^ 1, pf);  // plane ek + 1
    if (ek < ek_end) fetch(ek + 2, pf);
    aux_at(ek + 1, a_next);
    OwnT on{};
    if constexpr (OWN)
      if (owner && ek >= oz0) on = op.own_load(nst + (ek > ek0 ? plane : 0));
    __syncthreads();
    read_face(b ^ 1, F);
    if (ek > ek0) finish(ek - 1, b ^ 1);
    T tot[NC][4];
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        tot[c][q] = carry[c][q];
        carry[c][q] = T(0);
      }
    if (exy_ok && ek >= 0 && ek < G.nez) op.element(a, B, F, tot, carry);
    // node (ex + 1, ey + 1): corner x1 of this element and x0 of the next lane's
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const T s0 = (tot[c][0] + tot[c][1]) + lane_up(tot[c][0] - tot[c][1]);
      const T s1 = (tot[c][2] + tot[c][3]) + lane_up(tot[c][2] - tot[c][3]);
      pend[c] = s0 + s1;             // corner y1
      s_red[b][c][tid] = s0 - s1;    // corner y0, for the element row below
    }
    pown = op.own(B);
    po = on;
  };

  Face fa, fb;
  {
    Raw p0[NPF][NF];
    fetch(ek0, p0);
    fetch(ek0 + 1, pf);
    commit(0, p0);
  }
  Aux a_next{};
  aux_at(ek0, a_next);
  __syncthreads();
  read_face(0, fa);
  for (int ek = ek0; ek <= ek_end; ek += 2) {
    layer(ek, fa, fb, a_next);
    if (ek + 1 > ek_end) break;
    layer(ek + 1, fb, fa, a_next);
  }
  __syncthreads();
  finish(ek_end, (ek_end - ek0) & 1);
  if constexpr (RED) {
    __shared__ double s_rs[NT / 64];
    const double v = block_sum<NT>(racc, s_rs);
    if (tid == 0) op.partial(rslot, v);
  }
}
template <int TX, int TY, class Op>
__device__ __forceinline__ void march_modal(const Grid &G, const Op &op, int OZ, Blk3 b, int rslot = 0) {
  march_modal<TX, TY>(G, op, OZ, b.x, b.y, b.z, rslot);
}

}  // namespace vfg
