// FP32 stage 1 of one workgroup (owner-computes, blocked TwoSum accumulation) and the
// j-split form's reduce + FP64-master stage 2 of one body, shared by the stage-1 kernels
// (stage1.hip) and the paired backward kernels (adjoint.hip).  The kernel layout is
// described at the top of stage1.hip.
#pragma once

#include "grav_common.h"

namespace grav {
namespace {

// Knuth's TwoSum: hi + p == s + e exactly; hi <- s, lo <- lo + e.
__device__ __forceinline__ void two_sum_fold(float &hi, float &lo, float p) {
  const float s = hi + p;
  const float bp = s - hi;
  const float e = (hi - (s - bp)) + (p - bp);
  hi = s;
  lo += e;
}

// U j-bodies q[u] (indices j + u) against the K bodies of a lane, added in the order of u.
// PRIO: their rsq together at a raised wave priority (prio_up), taken by the loops of two and of
// four j-bodies per step.  MI355X, two per step, without and with it: 2^18 bodies with (1, 16)
// 16.38 and 15.51 ms; the j-split form at 16384 bodies 74.6 and 70.0 us, at 49999 605 and 569 us;
// the batched per-step schedule on 1024 universes of 32-2048 bodies 0.147 and 0.137 ms per step.
// One s_setprio pair per body instead of two bodies: 15.69 ms, 70.9 us, 573 us, 0.138 ms, and
// 1758 against 1746 us for the forward and backward of 128 such universes, whose last
// wavefronts run alone on their SIMDs.  The loop of eight serves launches of about one
// wavefront per SIMD, which it slows down (2000 bodies in 32 workgroups: a step of 36.7
// against 35.7 us).
template <int K, bool MASK, bool PRIO, int U>
__device__ __forceinline__ void pairs_f32(const float4 (&q)[U], const int j,
                                          const float (&xi)[K], const float (&yi)[K],
                                          const float (&zi)[K], const int (&ii)[K],
                                          const float eps2, float (&px)[K], float (&py)[K],
                                          float (&pz)[K]) {
  if constexpr (!PRIO && (U > 1 || K > 1)) {
    // pair by pair: written in the phases below, eight bodies' values stay alive together and
    // four bodies per lane take 243 VGPRs instead of 79
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const float4 qu[1] = {q[u]};
        const float x1[1] = {xi[k]}, y1[1] = {yi[k]}, z1[1] = {zi[k]};
        const int i1[1] = {ii[k]};
        float sx[1] = {px[k]}, sy[1] = {py[k]}, sz[1] = {pz[k]};
        pairs_f32<1, MASK, false>(qu, j + u, x1, y1, z1, i1, eps2, sx, sy, sz);
        px[k] = sx[0];
        py[k] = sy[0];
        pz[k] = sz[0];
      }
    return;
  }
  float dx[U][K], dy[U][K], dz[U][K], inv[U][K];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int k = 0; k < K; ++k) {
      dx[u][k] = q[u].x - xi[k];
      dy[u][k] = q[u].y - yi[k];
      dz[u][k] = q[u].z - zi[k];
      float r2 = __builtin_fmaf(dx[u][k], dx[u][k], eps2);
      r2 = __builtin_fmaf(dy[u][k], dy[u][k], r2);
      inv[u][k] = __builtin_fmaf(dz[u][k], dz[u][k], r2);
    }
  if constexpr (PRIO) prio_up();
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int k = 0; k < K; ++k) inv[u][k] = __builtin_amdgcn_rsqf(inv[u][k]);
  if constexpr (PRIO) prio_down();
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (MASK) inv[u][k] = (j + u == ii[k]) ? 0.0f : inv[u][k];
      const float s = (q[u].w * inv[u][k]) * (inv[u][k] * inv[u][k]);
      px[k] = __builtin_fmaf(dx[u][k], s, px[k]);
      py[k] = __builtin_fmaf(dy[u][k], s, py[k]);
      pz[k] = __builtin_fmaf(dz[u][k], s, pz[k]);
    }
}

// s_waitcnt immediate that waits for every scalar (and LDS) access and no other counter:
// vmcnt 63 (bits 3:0 and 15:14), expcnt 7 (6:4), lgkmcnt 0 (11:8).
constexpr unsigned kWaitScalar = 0xC07F;

// Accumulates j in [j0, j1) into the block partials px/py/pz, JB j-bodies per loop step (one
// s_load of JB float4).  The order of the pairs, hence the result, is the same for any JB.
// Two or four per step is the faster loop in launches of many workgroups, eight in smaller
// ones (pair_loop_width).  With one body per lane these loops run their loads one step ahead in
// two SGPR sets a and b: each half-step waits for the set it is about to use, issues the load of
// the other set's next step and only then computes, so the scalar load's latency hides
// behind a step of pairs (scalar loads can return out of order, so a wait is always for all
// of them; the explicit wait comes before the next load is issued).  MI355X, Plummer, two per
// step: 16.57-16.64 against 17.12-17.17 ms at 2^18 with (1, 16), the j-split form at 16384 bodies
// 0.079 against 0.081 ms, the batched per-step schedule on 4096 universes of 32-2048 bodies
// 0.548 against 0.563 ms per step (before the raised priority).  It made
// the j-split form with two bodies per lane slower (2^18: 18.7 against 17.4 ms), and with
// eight j-bodies per step the second set pushed SGPRs into VGPRs (K = 2: 51 to 118).
template <int K, bool MASK, int JB>
__device__ __forceinline__ void pair_range_f32(const float4 *__restrict__ posm, int j0, int j1,
                                               const float (&xi)[K], const float (&yi)[K],
                                               const float (&zi)[K], const int (&ii)[K],
                                               const float eps2, float (&px)[K],
                                               float (&py)[K], float (&pz)[K]) {
  int j = j0;
  if constexpr (JB <= 4 && K == 1) {
    if (j + JB <= j1) {
      float4 a[JB], b[JB];
#pragma unroll
      for (int u = 0; u < JB; ++u) a[u] = posm[j + u];
      for (; j + 2 * JB <= j1; j += 2 * JB) {
        __builtin_amdgcn_s_waitcnt(kWaitScalar);
#pragma unroll
        for (int u = 0; u < JB; ++u) b[u] = posm[j + JB + u];
        __builtin_amdgcn_sched_barrier(0);
        pairs_f32<K, MASK, (JB <= 4)>(a, j, xi, yi, zi, ii, eps2, px, py, pz);
        // the next step of set a, or (past the end) a step in range that is not used
        const int jn = min(j + 2 * JB, j1 - JB);
        __builtin_amdgcn_s_waitcnt(kWaitScalar);
#pragma unroll
        for (int u = 0; u < JB; ++u) a[u] = posm[jn + u];
        __builtin_amdgcn_sched_barrier(0);
        pairs_f32<K, MASK, (JB <= 4)>(b, j + JB, xi, yi, zi, ii, eps2, px, py, pz);
      }
      if (j + JB <= j1) {
        pairs_f32<K, MASK, (JB <= 4)>(a, j, xi, yi, zi, ii, eps2, px, py, pz);
        j += JB;
      }
    }
  } else {
    for (; j + JB <= j1; j += JB) {
      float4 q[JB];
#pragma unroll
      for (int u = 0; u < JB; ++u) q[u] = posm[j + u];
      pairs_f32<K, MASK, (JB <= 4)>(q, j, xi, yi, zi, ii, eps2, px, py, pz);
    }
  }
  for (; j < j1; ++j) {
    const float4 q[1] = {posm[j]};
    pairs_f32<K, MASK, (JB <= 4)>(q, j, xi, yi, zi, ii, eps2, px, py, pz);
  }
}

// Blocked compensated sum over j in [j0, j1).  MASK: the pairs with j in [ma, mb) (the
// workgroup's own i-range) run the self-masked pair routine.  That choice does not change a
// pair's value for j != i, and the blocks start at j0 whatever [ma, mb) is, so a body's sum
// does not depend on which i-tile holds it.
// fold(px, py, pz) takes each block's sums, in order.
template <int K, bool MASK, int JB, typename Fold>
__device__ __forceinline__ void sum_segment_f32(const float4 *__restrict__ posm, int j0, int j1,
                                                int jblock, int ma, int mb,
                                                const float (&xi)[K],
                                                const float (&yi)[K], const float (&zi)[K],
                                                const int (&ii)[K], const float eps2,
                                                Fold &&fold) {
  for (int jb = j0, je; jb < j1; jb = je) {
    je = (j1 - jb > jblock) ? jb + jblock : j1;  // no overflow for jblock near INT_MAX
    float px[K], py[K], pz[K];
#pragma unroll
    for (int k = 0; k < K; ++k) px[k] = py[k] = pz[k] = 0.0f;
    if constexpr (MASK) {
      const int a = min(je, max(jb, ma));
      const int b = max(a, min(je, mb));
      pair_range_f32<K, false, JB>(posm, jb, a, xi, yi, zi, ii, eps2, px, py, pz);
      pair_range_f32<K, true, JB>(posm, a, b, xi, yi, zi, ii, eps2, px, py, pz);
      pair_range_f32<K, false, JB>(posm, b, je, xi, yi, zi, ii, eps2, px, py, pz);
    } else {
      pair_range_f32<K, false, JB>(posm, jb, je, xi, yi, zi, ii, eps2, px, py, pz);
    }
    fold(px, py, pz);
  }
}

// Halves of the item-list forms (one body per lane).  A wavefront sums its j-range block after
// block of 256 bodies, so a batch of few universes lasts as long as the blocks of its largest one:
// 2048 bodies and four wavefronts, two blocks of 256 pairs that one wavefront alone issues at
// half the rate of two.  In halves a workgroup has a second set of wavefronts: each takes over the
// blocks of the second half of its counterpart's range and leaves their sums in LDS, and the
// first folds them in after its own in the same order, so the bits are those of one wavefront.
// A wavefront whose counterpart has one block or none ends at once.  Taken where there is a
// second block (up to 1024 j-bodies per wavefront, for the sums' LDS) and the launch is
// small: with wavefronts enough on every SIMD the second set gives nothing and costs its
// workgroups' slots.  So the limits count the first set's wavefronts, items times j_waves, on 1024
// SIMDs: six for steps, four for VJPs, whose workgroups hold more registers and LDS.  MI355X,
// eight launches without and with, us (wavefronts; universes of 64-2048 and 300-1000 bodies).
// Steps, one j-wave: 957 501 and 306, 2874 554 and 388, 6702 769 and 788; two: 3794 545 and 399,
// 5306 568 and 501, 7580 686 and 673; four: 4720 297 and 268, 7588 339 and 346, 10612 456 and 472.
// VJPs, one: 957 563 and 377, 2874 786 and 793; two: 1914 312 and 342, 2476 623 and 510, 3794 788
// and 735, 5748 688 and 750; four: 2360 320 and 275, 4720 474 and 512, 4952 442 and 486.
constexpr int kHalvesStepWaves = 6144;   // largest launches in halves, of steps
constexpr int kHalvesVjpWaves = 4096;    // and of VJPs
constexpr int kHalvesChunk = 1024;

// Whether the longest j-range of a wavefront has a second block and at most kHalvesChunk bodies.
inline bool halves_of(int max_bodies, int S) {
  const int chunk = ((max_bodies + S - 1) / S + 7) & ~7;
  return chunk > 256 && chunk <= kHalvesChunk;
}

// Block sums that a wavefront of the second set leaves at most: the blocks whose middle lies in
// the second half of a range of `chunk` bodies start in its last chunk / 2 + 128 bodies, and
// the VJP's own-tile segment divides them into three segments, each with a rounded-up number.
inline int half_slots(int max_bodies, int S) {
  const int chunk = ((max_bodies + S - 1) / S + 7) & ~7;
  return (chunk / 2 + 128) / 256 + 3;
}

// The FP64-master stage 2 of body i from its FP32 acceleration a, without contraction as
// k_stage2_f64m does it (v = a dt + v, r = v dt + r): r and v come as r64 and v64 hold them (stride
// n), the new ones go back there and the new FP32 position, with mass m, to out[i].
__device__ __forceinline__ void stage2_f64m_body(const float (&a)[3], double (&r)[3],
                                                 double (&v)[3], float m, float4 *out,
                                                 double *__restrict__ r64,
                                                 double *__restrict__ v64, int n, double dt,
                                                 int i) {
#pragma clang fp contract(off)
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    v[c] = static_cast<double>(a[c]) * dt + v[c];
    r[c] = v[c] * dt + r[c];
    v64[c * n + i] = v[c];
    r64[c * n + i] = r[c];
  }
  out[i] = make_float4(static_cast<float>(r[0]), static_cast<float>(r[1]),
                       static_cast<float>(r[2]), m);
}

// Where a fused step of the item-list form puts its results: the FP64 masters (stride m) and
// the new positions, which must not overlap the old ones.
struct StepIO {
  float4 *out;
  double *r64, *v64;
  double dt;
};

// The workgroup at (bx, by) of an (x, ny) grid owns i in [items[bx].x, items[bx].y) (at most
// 64*K bodies) against j in [items[bx].z, items[bx].w); items == NULL means one universe:
// i-tile bx of the shard [i0, i0 + m) against all n bodies, or, with diag_block > 0, against
// its own block of diag_block bodies only, or, with part != NULL, against the by-th of ny
// equal j-ranges of [0, n) (the j-split form: the workgroup writes its unscaled compensated
// partial to part[by][c][i - i0] in FP64, and a reduce kernel sums the ranges).  Outputs are
// rows i - i0 of (3, m) arrays; a whole universe is i0 = 0, m = n, and with items i0 = 0 and
// m is the row stride.  The item list lets one launch cover many universes (one item per
// universe tile).  JB: j-bodies per step of the pair loop (pair_range_f32), 2, 4 or 8; the
// result does not depend on it.  red: (S - 1) * 6 * (64 * K) floats of LDS.
// STEP (with items): instead of acc, the bodies' FP64-master stage 2 into io, bit for bit
// k_stage1_f32 followed by k_stage2_f64m.  With one body per lane the masters are loaded before
// the pair loop.
// HALVES = 2: 2 S wavefronts, see halves_of; slots is half_slots, and red is larger by
// S * slots * 3 * (64 * K) floats.
template <int K, int S, int JB, bool STEP = false, int HALVES = 1>
__device__ __forceinline__ void stage1_f32_block(const float4 *__restrict__ posm,
                                                 float *__restrict__ acc, int n, int i0, int m,
                                                 float G, float eps2, int mask_self,
                                                 int jblock,
                                                 const int4 *__restrict__ items,
                                                 int diag_block, double *__restrict__ part,
                                                 int bx, int by, int ny, float *red,
                                                 const StepIO io = StepIO{}, int slots = 0) {
  const int lane = threadIdx.x & (kWave - 1);
  const int any = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int half = HALVES == 2 && any >= S ? 1 : 0;
  const int wave = any - half * S;
  int ibase, iend, jlo, jhi;
  if (items != nullptr) {
    const int4 it = items[bx];
    ibase = it.x;
    iend = it.y;
    jlo = it.z;
    jhi = it.w;
  } else {
    ibase = i0 + bx * (kWave * K);
    iend = min(i0 + m, ibase + kWave * K);
    // diag_block > 0: only the i-tile's own block of diag_block bodies (a multiple of 64*K)
    jlo = diag_block > 0 ? (ibase / diag_block) * diag_block : 0;
    jhi = diag_block > 0 ? min(n, jlo + diag_block) : n;
    if (part != nullptr) {
      const int ns = ny;
      const int span = ((n + ns - 1) / ns + 7) & ~7;
      jlo = min(n, by * span);
      jhi = min(n, jlo + span);
    }
  }

  // This wave's j-range; with mask_self the pairs with j in the workgroup's own i-range
  // [ibase, iend) are self-masked.
  const int chunk = ((jhi - jlo + S - 1) / S + 7) & ~7;
  const int j0 = min(jhi, jlo + wave * chunk);
  const int j1 = min(jhi, j0 + chunk);
  if constexpr (HALVES == 2) {
    if (half != 0 && j1 - j0 <= jblock) return;   // one block or none: nothing to take over
  }

  float xi[K], yi[K], zi[K];
  int ii[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = ibase + k * kWave + lane;
    ii[k] = i;
    const float4 p = posm[min(i, iend - 1)];
    xi[k] = p.x;
    yi[k] = p.y;
    zi[k] = p.z;
  }

  double mr[3], mv[3];
  if constexpr (STEP && K == 1) {
    if (any == 0) {
      const int ic = min(ii[0], iend - 1);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        mr[c] = io.r64[c * m + ic];
        mv[c] = io.v64[c * m + ic];
      }
    }
  }

  float hx[K], hy[K], hz[K], lx[K], ly[K], lz[K];
#pragma unroll
  for (int k = 0; k < K; ++k) hx[k] = hy[k] = hz[k] = lx[k] = ly[k] = lz[k] = 0.0f;

  // eps2 in a VGPR, so that the first r2 FMA takes no SGPR operand (an SGPR operand adds
  // issue cycles to an FP32 instruction): 2^18 with (1, 16) 16.86 against 17.14 ms
  const float eps2v = in_vgpr(eps2);
  auto fold = [&](const float (&px)[K], const float (&py)[K], const float (&pz)[K]) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      two_sum_fold(hx[k], lx[k], px[k]);
      two_sum_fold(hy[k], ly[k], py[k]);
      two_sum_fold(hz[k], lz[k], pz[k]);
    }
  };
  const int ma = mask_self ? ibase : 0, mb = mask_self ? iend : 0;
  auto segment = [&](int a, int b, auto &&f) {
    if (mask_self)
      sum_segment_f32<K, true, JB>(posm, a, b, jblock, ma, mb, xi, yi, zi, ii, eps2v, f);
    else
      sum_segment_f32<K, false, JB>(posm, a, b, jblock, 0, 0, xi, yi, zi, ii, eps2v, f);
  };
  if constexpr (HALVES == 2) {
    const int blocks = (j1 - j0 + jblock - 1) / jblock;
    const int jm = min(j1, j0 + (blocks + 1) / 2 * jblock);
    float *h = red + (S - 1) * 6 * kWave * K + wave * slots * 3 * kWave * K + lane;
    if (half == 0) {
      segment(j0, jm, fold);
    } else {
      float *o = h;
      segment(jm, j1, [&](const float (&px)[K], const float (&py)[K], const float (&pz)[K]) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
          o[(3 * k) * kWave] = px[k];
          o[(3 * k + 1) * kWave] = py[k];
          o[(3 * k + 2) * kWave] = pz[k];
        }
        o += 3 * kWave * K;
      });
    }
    __syncthreads();
    if (half == 0) {
      for (int b = (blocks + 1) / 2; b < blocks; ++b, h += 3 * kWave * K) {
        float px[K], py[K], pz[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
          px[k] = h[(3 * k) * kWave];
          py[k] = h[(3 * k + 1) * kWave];
          pz[k] = h[(3 * k + 2) * kWave];
        }
        fold(px, py, pz);
      }
    }
    if constexpr (S == 1) {
      if (half != 0) return;
    }
  } else {
    segment(j0, j1, fold);
  }

  if constexpr (S > 1) {
    constexpr int L = kWave * K;
    if (wave > 0 && half == 0) {
      float *r = red + (wave - 1) * 6 * L;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int t = k * kWave + lane;
        r[0 * L + t] = hx[k];
        r[1 * L + t] = hy[k];
        r[2 * L + t] = hz[k];
        r[3 * L + t] = lx[k];
        r[4 * L + t] = ly[k];
        r[5 * L + t] = lz[k];
      }
    }
    __syncthreads();
    if (any != 0) return;
    // Not unrolled in a step of several bodies per lane: with every wavefront's sums loaded at
    // once (2, 8) and (4, 8) took 86 and 243 VGPRs instead of 50 and 79.  MI355X, a step of 1000
    // universes of 64-1024 bodies 88 and 71 us, 127 and 90 us.
#pragma unroll (STEP && K > 1 ? 1 : S)
    for (int w = 1; w < S; ++w) {
      const float *r = red + (w - 1) * 6 * L;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int t = k * kWave + lane;
        two_sum_fold(hx[k], lx[k], r[0 * L + t]);
        two_sum_fold(hy[k], ly[k], r[1 * L + t]);
        two_sum_fold(hz[k], lz[k], r[2 * L + t]);
        lx[k] += r[3 * L + t];
        ly[k] += r[4 * L + t];
        lz[k] += r[5 * L + t];
      }
    }
  }

  if (part != nullptr) {
    // hi + lo of two floats is exact in FP64
    double *o = part + static_cast<size_t>(by) * 3 * m;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int i = ii[k];
      if (i < iend) {
        o[i - i0] = static_cast<double>(hx[k]) + static_cast<double>(lx[k]);
        o[m + i - i0] = static_cast<double>(hy[k]) + static_cast<double>(ly[k]);
        o[2 * m + i - i0] = static_cast<double>(hz[k]) + static_cast<double>(lz[k]);
      }
    }
    return;
  }
  if constexpr (STEP) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int i = ii[k];
      if (i < iend) {
        const float a[3] = {G * (hx[k] + lx[k]), G * (hy[k] + ly[k]), G * (hz[k] + lz[k])};
        if constexpr (K != 1) {
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            mr[c] = io.r64[c * m + i];
            mv[c] = io.v64[c * m + i];
          }
        }
        stage2_f64m_body(a, mr, mv, posm[i].w, io.out, io.r64, io.v64, m, io.dt, i);
      }
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = ii[k];
    if (i < iend) {
      acc[i - i0] = G * (hx[k] + lx[k]);
      acc[m + i - i0] = G * (hy[k] + ly[k]);
      acc[2 * m + i - i0] = G * (hz[k] + lz[k]);
    }
  }
}

// The pair loop's j-bodies per step for a launch of `workgroups` workgroups of K bodies per
// lane; split: the j-split form.
//   * K = 1 from 256 workgroups: four, or two in the j-split form from 2048 workgroups.  MI355X,
//     two and four per step: owner-computes 16384 bodies 77.4 and 71.8 us, 2^18 15.39 and
//     15.20 ms; the batched per-step schedule on 1024 universes of 32-2048 bodies 1.387 and
//     1.348 ms per 10 steps; forward and backward of 4096 bodies over 60 steps (512 workgroups)
//     2.03 and 2.00 ms; but the j-split form at 16384 bodies (4096 workgroups) 70.2 and 70.8 us,
//     at 32768 248.8 and 251.2 us.  (Six: 70.8 us and 17.5 ms; eight, without loads ahead:
//     18.4 ms.)
//   * Fewer workgroups: eight.  One launch per universe of 32-2048 bodies (at most 32
//     workgroups) takes 38.3 ms per step of 4096 universes with two and 34.0 with eight.
//   * K = 2, plain loop: two from 1024 workgroups (2^18 bodies, (2, 16): 17.9 against 18.4 ms),
//     else eight.  From K = 4 eight always: the K registers of the i-bodies leave no room for
//     the shorter loop's gain.
inline int pair_loop_width(int64_t workgroups, int K, bool split) {
  if (K == 1) return workgroups < 256 ? 8 : split && workgroups >= 2048 ? 2 : 4;
  return (K >= 4 || workgroups < 1024) ? 8 : 2;
}

// sum over the j-ranges p of part[p][c][i] (C components a range), in FP64 and in range order,
// eight loads in flight.
template <int C>
__device__ __forceinline__ double split_sum(const double *__restrict__ part, int c, int i, int n,
                                            int splits) {
  const size_t stride = static_cast<size_t>(C) * n;
  const double *q = part + static_cast<size_t>(c) * n + i;
  double s = 0.0;
  int p = 0;
  for (; p + 8 <= splits; p += 8) {
    double v[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) v[t] = q[(p + t) * stride];
#pragma unroll
    for (int t = 0; t < 8; ++t) s += v[t];
  }
  for (; p < splits; ++p) s += q[p * stride];
  return s;
}

// Bodies of a workgroup of the reduce kernels of the fused steps, which give each component of
// a body a thread of its own: 64 bodies, one wavefront per component.  These kernels move little
// (4096 bodies, 8 ranges: 1 MB) and last as long as one thread's chain of loads, so they are
// spread over as many compute units as there are chunks of 64 bodies.
constexpr int kReduceBodies = kWave;

// Component c of body i in the reduce of the FP32 j-split form fused with the FP64-master stage
// 2: the acceleration is rounded to FP32 exactly as k_split_reduce<float> stores it, then r, v
// advance as in k_stage2_f64m (v = a dt + v, r = v dt + r, no contraction), so a step equals
// the two kernels' bit for bit without writing acc.  The new FP32 position (x, y, z, m) of
// body i goes to out[i], its mass with component 0; out may be in (no other thread touches them).
__device__ __forceinline__ void split_step_component(const double *__restrict__ part,
                                                     const float4 *in, float4 *out,
                                                     double *__restrict__ r64,
                                                     double *__restrict__ v64, int n, int splits,
                                                     double G, double dt, int c, int i) {
#pragma clang fp contract(off)
  const size_t at = static_cast<size_t>(c) * n + i;
  const double v0 = v64[at], r0 = r64[at];
  const float a32 = static_cast<float>(G * split_sum<3>(part, c, i, n, splits));
  const double v = static_cast<double>(a32) * dt + v0;
  const double r = v * dt + r0;
  v64[at] = v;
  r64[at] = r;
  float *o = reinterpret_cast<float *>(out + i);
  if (c == 0) o[3] = in[i].w;
  o[c] = static_cast<float>(r);
}

}  // namespace
}  // namespace grav
