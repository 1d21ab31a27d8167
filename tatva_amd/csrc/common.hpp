// Shared helpers: status/error plumbing, launch geometry, deterministic
// reductions.  Written for gfx950 (CDNA4): 64-wide wavefronts, 8 XCDs.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>

#include "../../include/tatva_amd.h"

namespace tatva {

void set_error(const std::string &msg);

#define TATVA_TRY_HIP(expr)                                                     \
  do {                                                                          \
    hipError_t _e = (expr);                                                     \
    if (_e != hipSuccess) {                                                     \
      ::tatva::set_error(std::string(#expr) + ": " + hipGetErrorString(_e));    \
      return TATVA_EHIP;                                                        \
    }                                                                           \
  } while (0)

#define TATVA_REQUIRE(cond, msg)                                                \
  do {                                                                          \
    if (!(cond)) {                                                              \
      ::tatva::set_error(msg);                                                  \
      return TATVA_EINVAL;                                                      \
    }                                                                           \
  } while (0)

#define TATVA_CHECK_LAUNCH()                                                    \
  do {                                                                          \
    hipError_t _e = hipGetLastError();                                          \
    if (_e != hipSuccess) {                                                     \
      ::tatva::set_error(std::string("kernel launch: ") + hipGetErrorString(_e)); \
      return TATVA_EHIP;                                                        \
    }                                                                           \
  } while (0)

constexpr int kWave = 64;
constexpr int kBlock = 256;
constexpr int kNumXcd = 8;
// Upper bound on blocks of a grid-stride reduction kernel: bounds the partials
// buffers and fixes the summation tree for a given problem size.
constexpr int kMaxReduceBlocks = 2048;

inline int reduce_grid(int64_t n, int threads_per_item = 1) {
  int64_t items = n * threads_per_item;
  int64_t b = (items + kBlock - 1) / kBlock;
  if (b < 1) b = 1;
  if (b > kMaxReduceBlocks) b = kMaxReduceBlocks;
  return (int)b;
}

inline int grid_for(int64_t n, int block = kBlock) {
  int64_t b = (n + block - 1) / block;
  return (int)(b < 1 ? 1 : b);
}

// Workgroups are dispatched round-robin over the 8 XCDs (block b -> XCD b % 8).
// Re-map so that each XCD walks one contiguous range of logical blocks: the
// neighbouring elements/rows it processes then share node data in its own L2.
__device__ __forceinline__ int64_t xcd_block(int b, int n) {
  const int xcd = b % kNumXcd;
  const int k = b / kNumXcd;
  const int q = n / kNumXcd;
  const int r = n % kNumXcd;
  return (int64_t)xcd * q + (xcd < r ? xcd : r) + k;
}

// Value of the lane that a DPP control pairs with this one (every lane active).
template <int CTRL>
__device__ __forceinline__ int dpp_move(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(dpp_move<CTRL>(__float_as_int(v)));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  return __hiloint2double(dpp_move<CTRL>(__double2hiint(v)), dpp_move<CTRL>(__double2loint(v)));
}
constexpr int kDppQuadFirst = 0x00;    // quad_perm [0, 0, 0, 0]
constexpr int kDppXor1 = 0xB1;         // quad_perm [1, 0, 3, 2]
constexpr int kDppXor2 = 0x4E;         // quad_perm [2, 3, 0, 1]
constexpr int kDppHalfMirror = 0x141;  // lane ^ 7 inside each group of 8
constexpr int kDppMirror = 0x140;      // lane ^ 15 inside each row of 16

__device__ __forceinline__ int read_lane(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float read_lane(float v, int lane) {
  return __int_as_float(read_lane(__float_as_int(v), lane));
}
__device__ __forceinline__ double read_lane(double v, int lane) {
  return __hiloint2double(read_lane(__double2hiint(v), lane), read_lane(__double2loint(v), lane));
}

// Sum over the wave in a fixed tree, the same value in every lane: rows of 16 by
// DPP, then the four rows as scalars (no LDS round trips, which each of the six
// steps of a shuffle tree takes; with the loads of sum_partials3 together the CG
// step of a 64^2 Poisson system went from 5.1 to 3.8 us, its SpMV from 5.1 to 4.4).
template <class T>
__device__ __forceinline__ T wave_sum(T v) {
  v += dpp_move<kDppXor1>(v);
  v += dpp_move<kDppXor2>(v);
  v += dpp_move<kDppHalfMirror>(v);
  v += dpp_move<kDppMirror>(v);
  return (read_lane(v, 0) + read_lane(v, 16)) + (read_lane(v, 32) + read_lane(v, 48));
}

// Deterministic block sum (fixed shuffle/LDS tree); result valid in thread 0.
template <class T>
__device__ __forceinline__ T block_sum(T v) {
  __shared__ T smem[kBlock / kWave];
  v = wave_sum(v);
  const int lane = threadIdx.x % kWave;
  const int wid = threadIdx.x / kWave;
  if (lane == 0) smem[wid] = v;
  __syncthreads();
  T s = T(0);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 0; w < kBlock / kWave; ++w) s += smem[w];
  }
  __syncthreads();
  return s;
}

// Deterministic block sum whose result every thread receives.
template <class T>
__device__ __forceinline__ T block_sum_all(T v) {
  __shared__ T smem[kBlock / kWave + 1];
  v = wave_sum(v);
  const int lane = threadIdx.x % kWave;
  const int wid = threadIdx.x / kWave;
  if (lane == 0) smem[wid] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    T s = T(0);
#pragma unroll
    for (int w = 0; w < kBlock / kWave; ++w) s += smem[w];
    smem[kBlock / kWave] = s;
  }
  __syncthreads();
  const T s = smem[kBlock / kWave];
  __syncthreads();
  return s;
}

// Sum of per-block partials written by an earlier kernel, in a fixed order;
// every thread receives the result.  Cross-block reductions go through a
// kernel boundary (which publishes the partials to every XCD) instead of an
// in-kernel device-scope fence and atomic: on CDNA4 with one L2 per XCD such a
// fence writes back the L2 and costs far more than re-reading a few KB of
// partials in each block.
template <class T>
__device__ __forceinline__ T sum_partials(const T *partials, int n) {
  T v = T(0);
  // (eight loads together; a load at a time, the loop waits for each)
  for (int i = threadIdx.x; i < n; i += 8 * kBlock) {
    T w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int j = i + k * kBlock;
      w[k] = partials[j < n ? j : 0];
      if (j >= n) w[k] = T(0);
    }
    v += ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
  }
  return block_sum_all(v);
}

// Three partial sums at once, one barrier: every thread adds the four wave
// sums itself in the same order, so all threads of all blocks get the same
// bits.  Call at most once per kernel (its LDS is not re-armed).
__device__ __forceinline__ void sum_partials3(const double *__restrict__ a, int na,
                                              const double *__restrict__ b, int nb,
                                              const double *__restrict__ c, int nc, double &sa,
                                              double &sb, double &sc) {
  __shared__ double sm[3][kBlock / kWave];
  // four values of each array per thread are loaded together (a load at a time,
  // the loops wait for one round trip each)
  const auto share = [](const double *__restrict__ p, int i, int n) {
    double v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int j = i + k * kBlock;
      v[k] = p[j < n ? j : 0];
      if (j >= n) v[k] = 0.0;
    }
    return (v[0] + v[1]) + (v[2] + v[3]);
  };
  double va = share(a, threadIdx.x, na), vb = share(b, threadIdx.x, nb),
         vc = share(c, threadIdx.x, nc);
  for (int i = threadIdx.x + 4 * kBlock; i < na; i += 4 * kBlock) va += share(a, i, na);
  for (int i = threadIdx.x + 4 * kBlock; i < nb; i += 4 * kBlock) vb += share(b, i, nb);
  for (int i = threadIdx.x + 4 * kBlock; i < nc; i += 4 * kBlock) vc += share(c, i, nc);
  va = wave_sum(va);
  vb = wave_sum(vb);
  vc = wave_sum(vc);
  const int lane = threadIdx.x % kWave;
  const int wid = threadIdx.x / kWave;
  if (lane == 0) {
    sm[0][wid] = va;
    sm[1][wid] = vb;
    sm[2][wid] = vc;
  }
  __syncthreads();
  sa = sb = sc = 0.0;
#pragma unroll
  for (int w = 0; w < kBlock / kWave; ++w) {
    sa += sm[0][w];
    sb += sm[1][w];
    sc += sm[2][w];
  }
}

// Two block sums at once (one barrier); results valid in thread 0.
__device__ __forceinline__ void block_sum2(double &a, double &b) {
  __shared__ double sm[2][kBlock / kWave];
  a = wave_sum(a);
  b = wave_sum(b);
  const int lane = threadIdx.x % kWave;
  const int wid = threadIdx.x / kWave;
  if (lane == 0) {
    sm[0][wid] = a;
    sm[1][wid] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double x = 0.0, y = 0.0;
#pragma unroll
    for (int w = 0; w < kBlock / kWave; ++w) {
      x += sm[0][w];
      y += sm[1][w];
    }
    a = x;
    b = y;
  }
}

// out[0] = sum (subtract == 0) or out[0] -= sum of partials[0..n): one block.
template <class T>
__global__ __launch_bounds__(kBlock) void k_finalize_sum(const T *__restrict__ partials, int n,
                                                         T *__restrict__ out, int subtract) {
  const T s = sum_partials(partials, n);
  if (threadIdx.x == 0) out[0] = subtract ? out[0] - s : s;
}

}  // namespace tatva
