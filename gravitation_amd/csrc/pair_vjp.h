// Vector-Jacobian product of the pair acceleration, shared by the single-universe and the
// batched adjoint kernels.
//
// Forward (per owner k): a_k = G sum_j m_j s_kj d_kj with d_kj = r_j - r_k,
// q = |d|^2 + eps^2, s = q^(-3/2).  Its adjoint against a cotangent field mu is
//   (J_r^T mu)_k = G sum_{j != k} T_kj w_kj,   T_kj = s (I - 3 d d^T / q),
//                  w_kj = m_k mu_j - m_j mu_k
//   (J_m^T mu)_k = -G sum_{j != k} s_kj d_kj . mu_j
// One pair costs 29 VALU ops + 1 v_rsq_f32 in FP32.  The caller adds G (and the step) once.
// The self pair (j == k) must go through the MASK path for every eps: w is formed with an FMA,
// so for j == k it would be the rounding error of m_k mu_k rather than exactly 0.
#pragma once

#include "grav_common.h"

namespace grav {

// Accumulates, for K owners per lane, the partials P += s (w - 3 (d.w)/q d) and
// Pg += s (d . mu_j) of U j-bodies (q = x, y, z, m; u = mu_j; indices j + t), in the order of t.
// PRIO: the rsq of the U * K pairs together at a raised wave priority (prio_up).
template <int K, bool MASK, bool PRIO, int U>
__device__ __forceinline__ void vjp_pairs(const float4 (&q)[U], const float4 (&u)[U],
                                          const int j, const float (&xk)[K],
                                          const float (&yk)[K], const float (&zk)[K],
                                          const float (&mk)[K], const float (&uxk)[K],
                                          const float (&uyk)[K], const float (&uzk)[K],
                                          const int (&kk)[K], const float eps2, float (&px)[K],
                                          float (&py)[K], float (&pz)[K], float (&pg)[K]) {
  float dx[U][K], dy[U][K], dz[U][K], iv[U][K];
#pragma unroll
  for (int t = 0; t < U; ++t)
#pragma unroll
    for (int k = 0; k < K; ++k) {
      dx[t][k] = q[t].x - xk[k];
      dy[t][k] = q[t].y - yk[k];
      dz[t][k] = q[t].z - zk[k];
      float r2 = __builtin_fmaf(dx[t][k], dx[t][k], eps2);
      r2 = __builtin_fmaf(dy[t][k], dy[t][k], r2);
      iv[t][k] = __builtin_fmaf(dz[t][k], dz[t][k], r2);
    }
  if constexpr (PRIO) prio_up();
#pragma unroll
  for (int t = 0; t < U; ++t)
#pragma unroll
    for (int k = 0; k < K; ++k) iv[t][k] = __builtin_amdgcn_rsqf(iv[t][k]);
  if constexpr (PRIO) prio_down();
#pragma unroll
  for (int t = 0; t < U; ++t)
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const float inv = (MASK && j + t == kk[k]) ? 0.0f : iv[t][k];
      const float inv2 = inv * inv;
      const float s = inv * inv2;
      const float wx = __builtin_fmaf(mk[k], u[t].x, -(q[t].w * uxk[k]));
      const float wy = __builtin_fmaf(mk[k], u[t].y, -(q[t].w * uyk[k]));
      const float wz = __builtin_fmaf(mk[k], u[t].z, -(q[t].w * uzk[k]));
      float dw = dx[t][k] * wx;
      dw = __builtin_fmaf(dy[t][k], wy, dw);
      dw = __builtin_fmaf(dz[t][k], wz, dw);
      const float c3 = (inv2 * dw) * 3.0f;
      px[k] = __builtin_fmaf(s, __builtin_fmaf(-c3, dx[t][k], wx), px[k]);
      py[k] = __builtin_fmaf(s, __builtin_fmaf(-c3, dy[t][k], wy), py[k]);
      pz[k] = __builtin_fmaf(s, __builtin_fmaf(-c3, dz[t][k], wz), pz[k]);
      float dm = dx[t][k] * u[t].x;
      dm = __builtin_fmaf(dy[t][k], u[t].y, dm);
      dm = __builtin_fmaf(dz[t][k], u[t].z, dm);
      pg[k] = __builtin_fmaf(s, dm, pg[k]);
    }
}

// One j-body.
template <int K, bool MASK>
__device__ __forceinline__ void vjp_pair(const float4 q, const float4 u, const int j,
                                         const float (&xk)[K], const float (&yk)[K],
                                         const float (&zk)[K], const float (&mk)[K],
                                         const float (&uxk)[K], const float (&uyk)[K],
                                         const float (&uzk)[K], const int (&kk)[K],
                                         const float eps2, float (&px)[K], float (&py)[K],
                                         float (&pz)[K], float (&pg)[K]) {
  const float4 q1[1] = {q}, u1[1] = {u};
  vjp_pairs<K, MASK, false>(q1, u1, j, xk, yk, zk, mk, uxk, uyk, uzk, kk, eps2, px, py, pz, pg);
}

// Knuth's TwoSum: hi + p == s + e exactly; hi <- s, lo <- lo + e.
__device__ __forceinline__ void two_sum_acc(float &hi, float &lo, float p) {
  const float s = hi + p;
  const float bp = s - hi;
  const float e = (hi - (s - bp)) + (p - bp);
  hi = s;
  lo += e;
}

}  // namespace grav
