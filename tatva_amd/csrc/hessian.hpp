// Colored Hessian rows straight from the mesh: a group of lanes takes one node,
// computes the rows of the element stiffness that belong to it from the node
// coordinates and the state, and decompresses them into CSR.
//
// For a quadrature point with weight w, material gradients B_a = dN_a/dX and
// spatial gradients b_a = F^-T B_a, the 3x3 block of nodes (a, b) is
//   Neo-Hookean        w [ mu (B_a . B_b) I + (mu - lambda ln J) b_b b_a^T + lambda b_a b_b^T ]
//   linear elasticity  w [ mu (B_a . B_b) I + mu B_b B_a^T + lambda B_a B_b^T ]
//   Poisson            w B_a . B_b
// (density.hpp's dP for the unit tangents e_k B_b, contracted with B_a), so a
// row costs a few products per column instead of one element Hessian-vector
// product per column.
//
// Against an element-stiffness buffer (one thread per column writing 4.6 kB per
// Hex8 element, one wave per matrix row gathering it): 64^3 Hex8 linear
// elasticity moved 2.4 GB through that buffer and took 633 + 1735 us; here
// each element's geometry is recomputed for each of its nodes and only the
// matrix is written: 396 us (656 MB, 1.7 TB/s).  48^3 Hex8 Neo-Hookean 1346
// -> 733 us, distorted linear elastic 1036 -> 344 us; 24^3 x 6 Tet4
// Neo-Hookean 193 -> 43 us; 200^2 Tri3 linear elastic 97 -> 15 us.  The sums are
// LDS adds one element after another: read, added and stored, each waiting for the
// element before, the same cases took 473, 820, 373, 52 and 16 us.  The rows of
// boxes are bound by their ~500 vector instructions a wave (half of the time) and
// 72 LDS adds (40%); a wave waits 60% of its life on its chain of loads, so six
// waves a SIMD matter (loading the next node's data under this one's work cost
// half of them: 505 us; forced to eight waves it spills: 628).  The Hex8 kernel
// of a general element holds 230-300 registers (two waves a SIMD, one for
// Neo-Hookean; forced to three it spills and runs twice as long).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "assembly.hpp"
#include "common.hpp"
#include "density.hpp"
#include "element.hpp"

namespace tatva {

// Lanes per node and per element.  Hex8: eight lanes an element (lane s takes
// quadrature points s, s + 8, ..., then one column block), 64 a node (the
// eight elements of an inner node at once).  Simplices: one lane an element;
// 32 lanes hold the ~24 tetrahedra of a node, 16 the ~6 triangles.
template <int KIND, int NC>
struct RowsShape {
  static constexpr int NNE = Elem<KIND>::NNE, D = Elem<KIND>::D, ND = NNE * NC;
  static constexpr int S = KIND == TATVA_HEX8 ? 8 : 1;
  static constexpr int LG = KIND == TATVA_HEX8 ? 64 : KIND == TATVA_TET4 ? 32 : 16;
  static constexpr int P = LG / S;  // elements of a node held at a time
  // entries per lane looked up ahead (an inner node's 27 / 15 / 7 neighbours);
  // elements whose blocks are read ahead of their sums
  static constexpr int kPre = (NC * NC * (KIND == TATVA_HEX8 ? 27 : KIND == TATVA_TET4 ? 15 : 7) + LG - 1) / LG;
  static constexpr int kAhead = KIND == TATVA_TET4 ? 6 : 3;
  // Hex8 stages the nodes' coordinates and state (general elements), simplices
  // their blocks and the blocks' colors
  static constexpr int kBlk = KIND == TATVA_HEX8 ? 64 * 6 : P * NC * ND;  // doubles
  static constexpr int kTab = KIND == TATVA_HEX8 ? 0 : P * ND;            // int32
  static __host__ __device__ size_t lds_bytes(int n_colors, bool staged) {
    return ((size_t)NC * (n_colors + 1) + (staged ? kBlk : 0)) * sizeof(double) +
           (((size_t)kTab * sizeof(int32_t) + 7) & ~size_t(7));
  }
};

// K block of (row node, column node) summed over one element's quadrature
// points, Hex8: every lane s of the element's eight computes the blocks of all
// eight columns at its points and the eight lanes exchange them so that lane s
// ends with column node s (sign index, hex_bin), out[c * NC + k].  xs: the
// element's staged nodes in sign order, 6 doubles each (X, u); ja: sign index
// of the row's node.  Columns are taken in the order j ^ s: lane s then keeps
// slots 0..3 and sends 4..7 to lane s ^ 7, whose slots 3..0 they are, and so
// on, with no selects; seen from lane s the element is mirrored in the
// directions of s's bits, which the signs t fold in.  ONE (a rule of one point): all
// eight lanes take it, each for its own column, with no exchange (32^3 Neo-Hookean,
// element order shuffled: 92 us, 212 with seven lanes' points left out by their weight;
// from the element stiffness, a buffer that the last-level cache holds, 186).
template <class Dens, bool ONE>
__device__ __forceinline__ void hex8_row_blocks(const double *__restrict__ xs, int ja,
                                                const QuadRule &quad, const Dens &dens, int s,
                                                double (&out)[Dens::NC * Dens::NC]) {
  constexpr int NC = Dens::NC, NV = NC * NC;
  const double t[3] = {(s & 1) ? -1.0 : 1.0, (s & 2) ? -1.0 : 1.0, (s & 4) ? -1.0 : 1.0};
  const double tdet = t[0] * t[1] * t[2];
  const int jr = ja ^ s;  // the row's node in this lane's order
#pragma unroll
  for (int i = 0; i < NV; ++i) out[i] = 0.0;
  for (int q0 = 0; q0 < quad.nq; q0 += 8) {
    const bool on = ONE || q0 + s < quad.nq;
    double x, y, z, wq;
    if constexpr (ONE) {
      x = quad.xi[0][0];
      y = quad.xi[0][1];
      z = quad.xi[0][2];
      wq = quad.w[0];
    } else {
      lane_point(quad, q0, s, x, y, z, wq);
    }
    x *= t[0];
    y *= t[1];
    z *= t[2];
    const HexPoint pt(x, y, z);
    double J[3][3] = {}, H[3][3] = {};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      double d[3];
      pt.dN(j, d);
      const double *nd = xs + (j ^ s) * 6;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double Xc = nd[c], Uc = Dens::kLinear ? 0.0 : nd[3 + c];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          J[k][c] += d[k] * Xc;
          if constexpr (!Dens::kLinear) H[k][c] += d[k] * Uc;
        }
      }
    }
    double inv[3][3];
    const double det = det_inv(J, inv);
    const double w = on ? tdet * det * wq : 0.0;
    // natural gradient of the row's node (jr is not a constant: by its signs)
    double da[3];
    {
      const double sx = (jr & 1) ? 1.0 : -1.0, sy = (jr & 2) ? 1.0 : -1.0, sz = (jr & 4) ? 1.0 : -1.0;
      da[0] = 0.125 * sx * (1.0 + sy * y) * (1.0 + sz * z);
      da[1] = 0.125 * sy * (1.0 + sx * x) * (1.0 + sz * z);
      da[2] = 0.125 * sz * (1.0 + sx * x) * (1.0 + sy * y);
    }
    double Ba[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) Ba[i] = inv[i][0] * da[0] + inv[i][1] * da[1] + inv[i][2] * da[2];
    double M[3][3], n[3], p[3], r[3];
    if constexpr (NC == 1 || !Dens::kLinear) {
      // w mu B_a . B_b as a natural covector on dN_b
      const double m = w * dens.modulus();
#pragma unroll
      for (int k = 0; k < 3; ++k)
        n[k] = m * (inv[0][k] * Ba[0] + inv[1][k] * Ba[1] + inv[2][k] * Ba[2]);
    }
    if constexpr (!Dens::kLinear) {
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) H[i][j] += J[i][j];
      const double detx = det_inv(H, M);
      const double c1 = w * dens.shear_modulus(detx / det), lm = w * dens.bulk_modulus();
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const double bi = M[i][0] * da[0] + M[i][1] * da[1] + M[i][2] * da[2];
        p[i] = c1 * bi;
        r[i] = lm * bi;
      }
    } else if constexpr (NC > 1) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        r[i] = w * Ba[i];
#pragma unroll
        for (int j = 0; j < 3; ++j) M[i][j] = inv[i][j];
      }
    }
    const auto block = [&](int j, double (&v)[NV]) {
      double d[3];
      pt.dN(j, d);
      if constexpr (NC == 1) {
        v[0] = n[0] * d[0] + n[1] * d[1] + n[2] * d[2];
      } else {
        double bb[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) bb[i] = M[i][0] * d[0] + M[i][1] * d[1] + M[i][2] * d[2];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            v[c * NC + k] = r[c] * bb[k];
            if constexpr (!Dens::kLinear) v[c * NC + k] += bb[c] * p[k];
          }
        if constexpr (!Dens::kLinear) {
          const double diag = n[0] * d[0] + n[1] * d[1] + n[2] * d[2];
#pragma unroll
          for (int c = 0; c < 3; ++c) v[c * NC + c] += diag;
        }
      }
    };
    if constexpr (ONE) {  // (slot 0 is the lane's own column)
      block(0, out);
      break;
    }
    // slot j + what the partner sends to it, over the three exchanges
    const auto half = [&](int j, double (&v)[NV]) {
      double send[NV];
      block(j, v);
      block(7 - j, send);
#pragma unroll
      for (int i = 0; i < NV; ++i) v[i] += dpp_move<kDppHalfMirror>(send[i]);
    };
    const auto quarter = [&](int j, double (&v)[NV]) {  // j in 0, 1
      double send[NV];
      half(j, v);
      half(j ^ 2, send);
#pragma unroll
      for (int i = 0; i < NV; ++i) v[i] += dpp_move<kDppXor2>(send[i]);
    };
    double v0[NV], v1[NV];
    quarter(0, v0);
    quarter(1, v1);
#pragma unroll
    for (int i = 0; i < NV; ++i) out[i] += v0[i] + dpp_move<kDppXor1>(v1[i]);
  }
  if constexpr (NC > 1 && Dens::kLinear) dens.row_block(out);
}

// The same for a simplex: one lane computes all column blocks of its element,
// out[c][b * NC + k].
template <int KIND, class Dens>
__device__ __forceinline__ void simplex_row_blocks(
    const double (&X)[Elem<KIND>::NNE][Elem<KIND>::D], const double (&ue)[Elem<KIND>::NNE][Dens::NC],
    int a, const QuadRule &quad, const Dens &dens,
    double (&out)[Dens::NC][Elem<KIND>::NNE * Dens::NC]) {
  constexpr int D = Elem<KIND>::D, NNE = Elem<KIND>::NNE, NC = Dens::NC;
  double B[D][NNE];
  const double det = simplex_geometry<D, NNE>(X, B);
  double w = 0.0;
  for (int q = 0; q < quad.nq; ++q) w += det * quad.w[q];
  double Ba[D], ba[D], b[D][NNE];
  double c1 = 0.0;
  if constexpr (!Dens::kLinear) {
    // spatial gradients from the current Jacobian J + dN u
    double A[D][D], inv[D][D];
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
      for (int j = 0; j < D; ++j) A[i][j] = (X[i + 1][j] - X[0][j]) + (ue[i + 1][j] - ue[0][j]);
    const double detx = det_inv(A, inv);
    c1 = w * dens.shear_modulus(detx / det);
#pragma unroll
    for (int i = 0; i < D; ++i) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < D; ++k) {
        b[i][k + 1] = inv[i][k];
        s -= inv[i][k];
      }
      b[i][0] = s;
    }
  }
#pragma unroll
  for (int i = 0; i < D; ++i) {
    Ba[i] = B[i][0];
    ba[i] = Dens::kLinear ? 0.0 : b[i][0];
#pragma unroll
    for (int k = 1; k < NNE; ++k) {
      Ba[i] = a == k ? B[i][k] : Ba[i];
      if constexpr (!Dens::kLinear) ba[i] = a == k ? b[i][k] : ba[i];
    }
  }
#pragma unroll
  for (int bn = 0; bn < NNE; ++bn) {
    if constexpr (NC == 1) {
      double e = 0.0;
#pragma unroll
      for (int i = 0; i < D; ++i) e += Ba[i] * B[i][bn];
      out[0][bn] = w * e;
    } else {
      double v[NC * NC];
      if constexpr (Dens::kLinear) {
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int k = 0; k < NC; ++k) v[c * NC + k] = w * Ba[c] * B[k][bn];
        dens.row_block(v);
      } else {
        double dot = 0.0;
#pragma unroll
        for (int i = 0; i < D; ++i) dot += Ba[i] * B[i][bn];
        const double diag = w * dens.modulus() * dot, lm = w * dens.bulk_modulus();
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int k = 0; k < NC; ++k)
            v[c * NC + k] = c1 * b[c][bn] * ba[k] + lm * ba[c] * b[k][bn] + (c == k ? diag : 0.0);
      }
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int k = 0; k < NC; ++k) out[c][bn * NC + k] = v[c * NC + k];
    }
  }
}

// Parallelepiped Hex8 elements and a tangent that does not depend on the state:
// the sum over quadrature points is det J  J^-1 M_ab J^-T with constants
// M_ab[k][l] = sum_q w_q dN_a/dxi_k dN_b/dxi_l (ref, laid out [k * 3 + l][a][b]
// over sign indices), so a lane computes its block without a point loop.  X:
// the lane's own node (sign index s); the Jacobian (linear coordinate modes)
// comes from sums and differences over the element's eight lanes.
template <class Dens>
__device__ __forceinline__ void hex8_affine_row_blocks(const double (&X)[3], int ja,
                                                       const double *__restrict__ ref,
                                                       const Dens &dens, int s,
                                                       double (&out)[Dens::NC * Dens::NC]) {
  constexpr int NC = Dens::NC;
  double m[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) m[i] = ref[i * 64 + ja * 8 + s];
  const bool b0 = s & 1, b1 = s & 2, b2 = s & 4;
  double J[3][3], inv[3][3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const auto diff = [](double v, double other, bool high) { return high ? v - other : other - v; };
    const double o1 = dpp_move<kDppXor1>(X[c]);
    const double s1 = X[c] + o1, d1 = diff(X[c], o1, b0);
    const double os = dpp_move<kDppXor2>(s1), od = dpp_move<kDppXor2>(d1);
    const double s12 = s1 + os, m1 = d1 + od, m2 = diff(s1, os, b1);
    J[0][c] = 0.125 * (m1 + dpp_move<kDppHalfMirror>(m1));
    J[1][c] = 0.125 * (m2 + dpp_move<kDppHalfMirror>(m2));
    J[2][c] = 0.125 * diff(s12, dpp_move<kDppHalfMirror>(s12), b2);
  }
  const double det = det_inv(J, inv);
  if constexpr (NC == 1) {
    double e = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int k = 0; k < 3; ++k)
        e += inv[i][k] * (m[k * 3] * inv[i][0] + m[k * 3 + 1] * inv[i][1] + m[k * 3 + 2] * inv[i][2]);
    out[0] = det * e;
  } else {
    double t[3][3];  // det J^-1 M
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int l = 0; l < 3; ++l)
        t[c][l] = det * (inv[c][0] * m[l] + inv[c][1] * m[3 + l] + inv[c][2] * m[6 + l]);
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int k = 0; k < 3; ++k)
        out[c * 3 + k] = t[c][0] * inv[k][0] + t[c][1] * inv[k][1] + t[c][2] * inv[k][2];
    dens.row_block(out);
  }
}

// The same for a box along the axes: the Jacobian is the diagonal of half the
// edges, so the block is det J M_ab[k][l] / (J_k J_l): fewer registers than the
// general parallelepiped's (six waves a SIMD instead of five, 64^3 linear elastic
// 433 -> 396 us).
template <class Dens>
__device__ __forceinline__ void hex8_box_row_blocks(const double (&X)[3], int ja,
                                                    const double *__restrict__ ref,
                                                    const Dens &dens, int s,
                                                    double (&out)[Dens::NC * Dens::NC]) {
  constexpr int NC = Dens::NC;
  double m[9];
#pragma unroll
  for (int i = 0; i < 9; ++i)
    if (NC > 1 || i % 4 == 0) m[i] = ref[i * 64 + ja * 8 + s];
  // (lane s ^ 7 is across the edge along z: its x and y are not looked at)
  const double o[3] = {dpp_move<kDppXor1>(X[0]), dpp_move<kDppXor2>(X[1]),
                       dpp_move<kDppHalfMirror>(X[2])};
  double J[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) J[c] = 0.5 * ((s >> c & 1) ? X[c] - o[c] : o[c] - X[c]);
  const double det = J[0] * J[1] * J[2], r = 1.0 / det;
  const double h[3] = {J[1] * J[2] * r, J[0] * J[2] * r, J[0] * J[1] * r};
  if constexpr (NC == 1) {
    out[0] = det * (h[0] * h[0] * m[0] + h[1] * h[1] * m[4] + h[2] * h[2] * m[8]);
  } else {
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int k = 0; k < 3; ++k) out[c * 3 + k] = det * h[c] * h[k] * m[c * 3 + k];
    dens.row_block(out);
  }
}

// k_node_rows on general Hex8 elements of a one-point rule.
constexpr int kGeomOnePoint = -1;

// p[0] += v on LDS.  A wave's LDS operations run in their order, so sums added one
// instruction after another have one order without a wait between them.
__device__ __forceinline__ void lds_add(double *p, double v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// One group of LG lanes per node.  The group's compressed Jacobian rows
// J[c][color] live in LDS (the last slot takes constrained columns); the
// node's elements are taken P at a time in ascending order, their blocks added to
// J one element after another (a simplex's block goes through LDS to all lanes of
// the group first), so the sums have one order where the columns of an element
// have colors of their own: a distance-2 coloring of a pattern that couples an
// element's dofs.  Only the last slot, which is never read, takes several
// columns of an element at once.  Then
// data[k] = J[c][colors[indices[k]]] (sparse/base.py:173).
// The loads are issued level by level (the node's rows and elements, their row
// ranges and element nodes, column indices and node data, colors), none behind
// a branch: a lane without work reads a valid address and drops the value.
// Behind branches each load waited for the one before (64^3 Hex8 linear
// elasticity, general geometry: 1540 us against 1130 us).
template <int KIND, class Dens, int GEOM, bool MAPPED>
__global__ __launch_bounds__(kBlock) void k_node_rows(
    int64_t n_nodes, int64_t n_rows, const double *__restrict__ coords,
    const int32_t *__restrict__ conn, QuadRule quad, const double *__restrict__ ref, Dens dens,
    const double *__restrict__ u, const int32_t *__restrict__ dof_map,
    const int32_t *__restrict__ colors, int n_colors, const int32_t *__restrict__ indptr,
    const int32_t *__restrict__ indices, const int32_t *__restrict__ inv_ptr,
    const int32_t *__restrict__ inv_list, double *__restrict__ data) {
  using Sh = RowsShape<KIND, Dens::NC>;
  constexpr int NNE = Sh::NNE, D = Sh::D, NC = Dens::NC, ND = Sh::ND, S = Sh::S, LG = Sh::LG,
                P = Sh::P;
  constexpr bool kHex = KIND == TATVA_HEX8;
  constexpr int NL = kHex ? 1 : NNE;  // nodes a lane loads
  constexpr bool ONE = GEOM == kGeomOnePoint;
  constexpr bool AFFINE = GEOM != kGeomGeneral && !ONE;
  static_assert(!AFFINE || (kHex && Dens::kLinear), "constant blocks");
  static_assert(!ONE || kHex, "simplices take one lane an element");
  extern __shared__ unsigned char lds_raw[];
  const int lane = threadIdx.x % LG;
  const int pl = lane / S, s = lane % S;
  const int64_t node =
      xcd_block(blockIdx.x, gridDim.x) * (blockDim.x / LG) + threadIdx.x / LG;
  if (node >= n_nodes) return;
  unsigned char *mine = lds_raw + (size_t)(threadIdx.x / LG) * Sh::lds_bytes(n_colors, !AFFINE);
  const int ncol = n_colors + 1;
  double *Jr = reinterpret_cast<double *>(mine);
  double *blk = Jr + (size_t)NC * ncol;
  int32_t *ctab = reinterpret_cast<int32_t *>(blk + Sh::kBlk);
  // level 1: the node's rows and element range
  int32_t row[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) row[c] = MAPPED ? dof_map[node * NC + c] : (int32_t)(node * NC + c);
  const int32_t b0 = inv_ptr[node], b1 = inv_ptr[node + 1];
  // level 2: row ranges, this lane's element.  The rows' entries are flattened:
  // entry t of the group is data[at + t] of row c, off <= t < the next off.
  const auto element_of = [&](int32_t p0) -> int32_t {
    return inv_list[pl < b1 - p0 ? p0 + pl : p0 < b1 ? p0 : 0];
  };
  int32_t k0[NC], off1[NC];  // start of each row, end of its entries
  int32_t total = 0;
  int32_t packed = element_of(b0);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int32_t r = row[c] >= 0 && row[c] < n_rows ? row[c] : 0;
    k0[c] = indptr[r];
    off1[c] = indptr[r + 1];
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int32_t len = row[c] >= 0 && row[c] < n_rows ? off1[c] - k0[c] : 0;
    k0[c] -= total;
    total += len;
    off1[c] = total;
  }
  if (total == 0) return;
  // (sums instead of selects: selects over these arrays end in scratch memory)
  const auto row_of = [&](int t) -> int {
    int c = 0;
#pragma unroll
    for (int i = 0; i + 1 < NC; ++i) c += int(t >= off1[i]);
    return c;
  };
  const auto entry = [&](int t) -> int32_t {
    int32_t k = k0[0] + t;
#pragma unroll
    for (int i = 1; i < NC; ++i) k += int(t >= off1[i - 1]) * (k0[i] - k0[i - 1]);
    return k;
  };
  // level 3: the columns of this lane's first entries, the element's nodes
  int32_t pre[Sh::kPre];
#pragma unroll
  for (int i = 0; i < Sh::kPre; ++i) {
    const int t = lane + i * LG;
    pre[i] = indices[entry(t < total ? t : 0)];
  }
  int32_t g[NL];
  const auto nodes_of = [&](int32_t pk) {
    const int32_t *c = conn + (int64_t)(pk >> 3) * NNE;
    if constexpr (kHex) {
      g[0] = c[hex_bin(s)];  // lane s takes the node of sign index s
    } else {
#pragma unroll
      for (int i = 0; i < NL; ++i) g[i] = c[i];
    }
  };
  nodes_of(packed);
  // level 4: colors of those columns (used at the end)
#pragma unroll
  for (int i = 0; i < Sh::kPre; ++i) pre[i] = colors[pre[i]];
  for (int i = lane; i < NC * ncol; i += LG) Jr[i] = 0.0;
  wave_lds_sync();  // the lanes add to entries that others have zeroed
  for (int32_t p0 = b0; p0 < b1; p0 += P) {
    const int cnt = b1 - p0 < P ? b1 - p0 : P;
    const int a = packed & 7;
    const Dens de = dens.at(packed >> 3);
    // level 4: node data
    double X[NL][D], ue[NL][NC];
    int32_t sd[NL * NC], col[NL * NC];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        const int64_t dof = (int64_t)g[i] * NC + k;
        sd[i * NC + k] = MAPPED ? dof_map[dof] : (int32_t)dof;
        ue[i][k] = Dens::kLinear ? 0.0 : u[dof];
      }
#pragma unroll
      for (int j = 0; j < D; ++j) X[i][j] = coords[(int64_t)g[i] * D + j];
    }
#pragma unroll
    for (int i = 0; i < NL * NC; ++i) {
      const int32_t k = colors[sd[i] >= 0 ? sd[i] : 0];
      col[i] = sd[i] >= 0 ? k : n_colors;
    }
    // the next chunk's elements and nodes
    if (p0 + P < b1) {
      packed = element_of(p0 + P);
      nodes_of(packed);
    }
    if constexpr (kHex) {
      double v[NC * NC];
      if constexpr (GEOM == kGeomBox) {
        hex8_box_row_blocks<Dens>(X[0], hex_bin(a), ref, de, s, v);
      } else if constexpr (AFFINE) {
        hex8_affine_row_blocks<Dens>(X[0], hex_bin(a), ref, de, s, v);
      } else {
#pragma unroll
        for (int j = 0; j < 3; ++j) blk[lane * 6 + j] = X[0][j];
        if constexpr (!Dens::kLinear) {
#pragma unroll
          for (int j = 0; j < 3; ++j) blk[lane * 6 + 3 + j] = ue[0][j];
        }
        wave_lds_sync();
        hex8_row_blocks<Dens, ONE>(blk + pl * 48, hex_bin(a), quad, de, s, v);
        wave_lds_sync();  // the staged nodes have been read
      }
      // element after element, its eight lanes adding their blocks
      for (int p = 0; p < cnt; ++p)
        if (pl == p) {
#pragma unroll
          for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int k = 0; k < NC; ++k) lds_add(Jr + c * ncol + col[k], v[c * NC + k]);
        }
    } else {
      double v[NC][ND];
      simplex_row_blocks<KIND, Dens>(X, ue, a, quad, de, v);
      wave_lds_sync();  // the blocks of the chunk before have been read
#pragma unroll
      for (int i = 0; i < ND; ++i) ctab[pl * ND + i] = col[i];
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < ND; ++i) blk[(pl * NC + c) * ND + i] = v[c][i];
      wave_lds_sync();
      // element after element, its values taken by the group's lanes; those of
      // some elements are read ahead of their sums
      constexpr int R = (NC * ND + LG - 1) / LG, W = Sh::kAhead;
      for (int pb = 0; pb < cnt; pb += W) {
        double val[W][R];
        int32_t dst[W][R];
#pragma unroll
        for (int pi = 0; pi < W; ++pi)
#pragma unroll
          for (int rr = 0; rr < R; ++rr) {
            const int p = pb + pi < cnt ? pb + pi : 0;
            const int i = rr * LG + lane < NC * ND ? rr * LG + lane : 0;
            const int c = i / ND, j = i - c * ND;
            val[pi][rr] = blk[p * NC * ND + i];
            dst[pi][rr] = c * ncol + ctab[p * ND + j];
          }
#pragma unroll
        for (int pi = 0; pi < W; ++pi) {
          if (pb + pi >= cnt) break;
#pragma unroll
          for (int rr = 0; rr < R; ++rr)
            if (rr * LG + lane < NC * ND) lds_add(Jr + dst[pi][rr], val[pi][rr]);
        }
      }
    }
  }
  wave_lds_sync();
#pragma unroll
  for (int i = 0; i < Sh::kPre; ++i) {
    const int t = lane + i * LG;
    if (t < total) data[entry(t)] = Jr[row_of(t) * ncol + pre[i]];
  }
  for (int t = lane + Sh::kPre * LG; t < total; t += LG) {
    const int32_t k = entry(t);
    data[k] = Jr[row_of(t) * ncol + colors[indices[k]]];
  }
}

}  // namespace tatva
