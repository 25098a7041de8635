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
// PRIO: the rsq of the U * K pairs together at a raised wave priority (prio_up).  Without it pair
// by pair: in phases, two and four bodies per lane took 94 and 168 VGPRs instead of 59 and 126
// and lost wavefronts.  MI355X, in phases and pair by pair: a quarter of the rows of 65536
// bodies with (2, 8) 1787 and 1677 us, the j-split VJP of 16384 with (2, 4) in 4 ranges 234 and 225
// us, of 65536 with (2, 2) in 8 ranges 3.36 and 3.12 ms.  (The other way round where the grid left
// the wavefronts unused: 40000 with (2, 2) 1.22 and 1.39 ms.)
template <int K, bool MASK, bool PRIO, int U>
__device__ __forceinline__ void vjp_pairs(const float4 (&q)[U], const float4 (&u)[U],
                                          const int j, const float (&xk)[K],
                                          const float (&yk)[K], const float (&zk)[K],
                                          const float (&mk)[K], const float (&uxk)[K],
                                          const float (&uyk)[K], const float (&uzk)[K],
                                          const int (&kk)[K], const float eps2, float (&px)[K],
                                          float (&py)[K], float (&pz)[K], float (&pg)[K]) {
  if constexpr (!PRIO && (U > 1 || K > 1)) {
#pragma unroll
    for (int t = 0; t < U; ++t)
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const float4 q1[1] = {q[t]}, u1[1] = {u[t]};
        const float x1[1] = {xk[k]}, y1[1] = {yk[k]}, z1[1] = {zk[k]}, m1[1] = {mk[k]};
        const float ux1[1] = {uxk[k]}, uy1[1] = {uyk[k]}, uz1[1] = {uzk[k]};
        const int k1[1] = {kk[k]};
        float sx[1] = {px[k]}, sy[1] = {py[k]}, sz[1] = {pz[k]}, sg[1] = {pg[k]};
        vjp_pairs<1, MASK, false>(q1, u1, j + t, x1, y1, z1, m1, ux1, uy1, uz1, k1, eps2, sx, sy,
                                  sz, sg);
        px[k] = sx[0];
        py[k] = sy[0];
        pz[k] = sz[0];
        pg[k] = sg[0];
      }
    return;
  }
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
