// Jacobi-PCG state shared by the single-solve and batched solvers.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "common.hpp"
#include "mesh.hpp"

namespace tatva {

// Device-side record of one solve; block 0 of the last kernel of an
// iteration writes it, the host reads it between launches.
struct PcgState {
  double rr;
  double bb;
  double tol2;
  int iter;
  int done;
  int status;
  int maxiter;
  // single-reduction CG: alpha_i, gamma_i and the iteration count written by
  // the step kernel of parity q = i mod 2 and read at parity q ^ 1
  double alpha[2];
  double gamma[2];
  int it[2];
  // FP32 matrix-free CG: the p and x update of iteration i, written by its
  // step kernel (slot i mod 2) and applied by the next operator launch
  CgDeferCoef defer[2];
};

// Vector kernels use at most this many blocks (4 per CU): the partials each
// block re-sums stay a few KB.
constexpr int kVecBlocks = 1024;

inline int vec_grid(int64_t n) {
  int64_t b = (n + kBlock - 1) / kBlock;
  if (b < 1) b = 1;
  if (b > kVecBlocks) b = kVecBlocks;
  return (int)b;
}

// Grid of a CG step kernel whose threads load `per_thread` elements before
// summing the shares of the previous step, and of the kernels that write
// those shares.  Every step block sums all of them, so the grid is no larger
// than the prefetch needs: enough blocks for the prefetched elements to cover
// n, at least one block per CU (fewer only when n gives fewer blocks of one
// element per thread), at most kVecBlocks.
constexpr int kStepMinBlocks = 256;

inline int step_grid(int64_t n, int per_thread) {
  const int64_t per_block = (int64_t)kBlock * per_thread;
  const int64_t lo = std::min<int64_t>(kStepMinBlocks, vec_grid(n));
  return (int)std::min<int64_t>(kVecBlocks, std::max(lo, (n + per_block - 1) / per_block));
}

// KB of the FP32 matrix-free form (solver_kernels.hip) by nodes, block `block` of
// n_blocks of a solve that is not done: single solves on Hex8 meshes and every
// slot of a batch.  w = H z is
// summed here from the tiles' slots (ascending tile) instead of by a gather
// kernel of its own: the tile kernel's shares give w.u, so nothing needs w before
// the scalars are known, and w is neither written nor read back.  dof_map: the
// vectors are reduced (an index outside [0, n) is skipped), or NULL: full-length,
// D^-1 = 0 on the dofs outside the system.
// kDefer: p and x are left to the next operator launch (their coefficients go to
// st->defer[q]; x and p are not touched and may be NULL), and the new z goes to z
// while that launch still reads the old one from the other buffer.
// A thread takes kStepNodes nodes at a time (a stride apart), loaded before the
// scalars are summed, their slot lists walked side by side.  Four consecutive
// nodes in 16-byte vectors measured no faster (105 against 102 us at 160^3),
// non-temporal stores slower (124 us: a thread's 12 bytes are no whole line).
constexpr int kStepNodes = 2;

template <int NC, bool kDefer>
__device__ __forceinline__ void node_step(
    int block, int n_blocks, int64_t n_nodes, int64_t n, const int32_t *__restrict__ slot_ptr,
    const float *__restrict__ partial, const int32_t *__restrict__ dof_map, float *__restrict__ x,
    float *__restrict__ r, float *__restrict__ z, float *__restrict__ p, float *__restrict__ s,
    const float *__restrict__ dinv, const double *__restrict__ part_delta, int n_delta,
    const double *__restrict__ part_g_old, const double *__restrict__ part_rr_old, int n_old,
    double *__restrict__ part_g_new, double *__restrict__ part_rr_new, int q,
    PcgState *__restrict__ st) {
  const int iter = st->it[q ^ 1];
  constexpr int K = kStepNodes, M = K * NC;
  const int64_t stride = (int64_t)n_blocks * kBlock;
  struct Nodes {
    float w[M], s[M], r[M], d[M], z[M], p[M], x[M];
    int64_t at[M];  // -1: nothing to write
  };
  const auto load = [&](int64_t i, Nodes &N) {
    int32_t b[K], len[K], longest = 0;
    // (past the end the last node again, and nothing written)
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int64_t node = i + k * stride;
      const int64_t g = node < n_nodes ? node : n_nodes - 1;
      b[k] = slot_ptr[g];
      len[k] = slot_ptr[g + 1];
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int64_t dof = g * NC + c;
        const int64_t at = dof_map ? (int64_t)dof_map[dof] : dof;
        N.at[k * NC + c] = at >= 0 && at < n ? at : -1;
      }
    }
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const int64_t at = N.at[j] >= 0 ? N.at[j] : 0;
      N.s[j] = s[at];
      N.r[j] = r[at];
      N.d[j] = dinv[at];
      if constexpr (!kDefer) {
        N.z[j] = z[at];
        N.p[j] = p[at];
        N.x[j] = x[at];
      }
      if (i + (j / NC) * stride >= n_nodes) N.at[j] = -1;
      N.w[j] = 0.0f;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      len[k] -= b[k];
      longest = max(longest, len[k]);
    }
    for (int32_t j = 0; j < longest; ++j)
#pragma unroll
      for (int k = 0; k < K; ++k)
        if (j < len[k]) {
          const float *src = partial + (int64_t)(b[k] + j) * NC;
#pragma unroll
          for (int c = 0; c < NC; ++c) N.w[k * NC + c] += src[c];
        }
  };
  const int64_t i0 = (int64_t)block * kBlock + threadIdx.x;
  Nodes pre;
  load(i0, pre);
  double gamma, rr, delta;
  sum_partials3(part_g_old, n_old, part_rr_old, n_old, part_delta, n_delta, gamma, rr, delta);
  const bool first = iter == 0;
  const double beta = first ? 0.0 : gamma / st->gamma[q ^ 1];
  const double denom = first ? delta : delta - beta * gamma / st->alpha[q ^ 1];
  const bool converged = rr <= st->tol2;
  const bool spent = iter >= st->maxiter;
  const bool bad = !(denom > 0.0) || !isfinite(denom) || !isfinite(gamma) || !isfinite(rr);
  if (converged || spent || bad) {
    if (block == 0 && threadIdx.x == 0) {
      st->done = 1;
      st->rr = rr;
      st->iter = iter;
      st->status = converged ? TATVA_OK : spent ? TATVA_ENOTCONV : TATVA_EBREAKDOWN;
    }
    return;
  }
  const double alpha = gamma / denom;
  const float a = float(alpha), bt = float(beta);
  if (block == 0 && threadIdx.x == 0) {
    st->alpha[q] = alpha;
    st->gamma[q] = gamma;
    st->it[q] = iter + 1;
    st->iter = iter + 1;
    st->rr = rr;
    if constexpr (kDefer) st->defer[q] = CgDeferCoef{a, bt, first ? 1 : 2, 0};
  }
  double sg = 0.0, srr = 0.0;
  // the expressions of k_cg_step (p and s hold no values before iteration 0)
  const auto update = [&](const Nodes &N) {
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const int64_t k = N.at[j];
      if (k < 0) continue;
      if constexpr (!kDefer) {
        const float pn = first ? N.z[j] : N.z[j] + bt * N.p[j];
        p[k] = pn;
        x[k] = N.x[j] + a * pn;
      }
      const float sn = first ? N.w[j] : N.w[j] + bt * N.s[j];
      const float rn = N.r[j] - a * sn;
      const float zn = N.d[j] * rn;
      s[k] = sn;
      r[k] = rn;
      z[k] = zn;
      sg += (double)rn * (double)zn;
      // D^-1 = 0 marks a dof outside the system: its r is not part of the residual
      srr += N.d[j] != 0.0f ? (double)rn * (double)rn : 0.0;
    }
  };
  update(pre);
  for (int64_t i = i0 + K * stride; i < n_nodes; i += K * stride) {
    Nodes N;
    load(i, N);
    update(N);
  }
  block_sum2(sg, srr);
  if (threadIdx.x == 0) {
    part_g_new[block] = sg;
    part_rr_new[block] = srr;
  }
}

// Matrix-free FP32 PCG set-up on stream s: st reset, dinv = 1/diag,
// r = b - H(u) x, p = D^-1 r, the shares of r.z (into part_rz1), r.r
// (part_rr1) and b.b over gv blocks, and the state (tol, maxiter, done when
// b == 0 or r already small).  lin: the density's cached linearisation at u
// (launch_linearize_f32), or NULL to linearise in the product; geo: an affine
// Hex8 mesh's geometry cache (launch_geometry_cache_f32), or NULL.  diag_map:
// the vectors are full-length and diag is the reduced diagonal (n_red entries)
// read through this dof map (dinv = 0 outside the system), or NULL: diag is n
// long.
int matfree_pcg_setup(tatva_mesh *m, const tatva_density *d, const float *u,
                      const int32_t *dof_map, int64_t n, const float *diag, const float *b,
                      const float *x, float *r, float *p, float *Ap, float *dinv,
                      double *part_rz1, double *part_rr1, double *part_bb, int gv, double tol,
                      int maxiter, PcgState *st, hipStream_t s, const float *lin = nullptr,
                      const float *geo = nullptr, const int32_t *diag_map = nullptr,
                      int64_t n_red = 0);

}  // namespace tatva
