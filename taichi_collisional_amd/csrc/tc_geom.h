// Smallest enclosing ball, computed by one wave or one block (device side of
// the cell geometry of P2M / M2M, taichi_with_jerks/kernel_fast_lean.h:733-763
// and :875-935, which use the Miniball of miniball.hpp).
//
// Algorithm (same as the CPU oracle, so both produce the same ball up to
// rounding; the minimum ball is unique): start from point 0; repeatedly find
// the point of largest excess |q-c|^2 - r^2 (threads scan subsets, then an
// argmax with ties to the lowest index); if it lies outside, the new ball is the smallest ball of
// (support set + q) with q on its boundary, found by testing the circumball of
// q with every subset of the support (<= 15 candidates, each of <= 4 points).
// The radius grows strictly, so the loop ends; the final ball encloses every
// point and is the minimum ball of its own support, hence of all points.
// Every thread runs the small solves on identical data, so the result is
// uniform across the block.  Contraction is off to match the CPU oracle.
#pragma once
#include "tc_common.h"

namespace tcfmm {

struct DBall {
  double c[3];
  double r2;
};

// Candidate masks of a refinement step: lane l < 16 tries the support points
// whose bits are set in l (at most three).  slot[i]: the i-th of them, 4 where
// there is none.
struct BallLane {
  int slot[3], count;
};
__device__ __forceinline__ BallLane ball_lane(int lane) {
  BallLane t = {{4, 4, 4}, 0};
#pragma unroll
  for (int s = 0; s < 4; s++)
    if (lane & (1 << s)) {
      if (t.count == 0) t.slot[0] = s;
      if (t.count == 1) t.slot[1] = s;
      if (t.count == 2) t.slot[2] = s;
      t.count++;
    }
  return t;
}

// Candidate `lane` of one refinement step: the smallest ball with bq and the
// lane's support points on its boundary (the circumcentre in their affine
// hull), valid when it also holds the other support points.
//
// One straight path for one to four points, so that the lanes' different
// candidates run side by side: a missing point is bq itself (its edge vector
// is zero) and its row of the Gram matrix the unit row, with which the 3 x 3
// solution takes, bit for bit, the values of the smaller system.
__device__ __forceinline__ bool candidate_ball(int lane, const BallLane &t, int ns,
                                               const double (&bq)[3], const double (&sup)[4][3],
                                               DBall &cb) {
#pragma clang fp contract(off)
  double v[3][3], A[3][3], rhs[3];
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int d = 0; d < 3; d++) {
      double p = bq[d];
#pragma unroll
      for (int s = i; s < 4; s++) p = t.slot[i] == s ? sup[s][d] : p;
      v[i][d] = p - bq[d];
    }
#pragma unroll
  for (int i = 0; i < 3; i++) {
#pragma unroll
    for (int j = 0; j <= i; j++)
      A[i][j] = A[j][i] = v[i][0] * v[j][0] + v[i][1] * v[j][1] + v[i][2] * v[j][2];
    rhs[i] = 0.5 * A[i][i];
    A[i][i] = i < t.count ? A[i][i] : 1.0;
  }
  const double c00 = A[1][1] * A[2][2] - A[1][2] * A[2][1];
  const double c01 = A[1][2] * A[2][0] - A[1][0] * A[2][2];
  const double c02 = A[1][0] * A[2][1] - A[1][1] * A[2][0];
  const double det = A[0][0] * c00 + A[0][1] * c01 + A[0][2] * c02;
  bool ok = lane < (1 << ns) && t.count <= 3 &&
            fabs(det) > 1e-13 * A[0][0] * A[1][1] * A[2][2];
  double inv[3][3];
  inv[0][0] = c00;
  inv[0][1] = A[0][2] * A[2][1] - A[0][1] * A[2][2];
  inv[0][2] = A[0][1] * A[1][2] - A[0][2] * A[1][1];
  inv[1][0] = c01;
  inv[1][1] = A[0][0] * A[2][2] - A[0][2] * A[2][0];
  inv[1][2] = A[0][2] * A[1][0] - A[0][0] * A[1][2];
  inv[2][0] = c02;
  inv[2][1] = A[0][1] * A[2][0] - A[0][0] * A[2][1];
  inv[2][2] = A[0][0] * A[1][1] - A[0][1] * A[1][0];
  double lam[3];
#pragma unroll
  for (int i = 0; i < 3; i++)
    lam[i] = (inv[i][0] * rhs[0] + inv[i][1] * rhs[1] + inv[i][2] * rhs[2]) / det;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    double c = bq[d];
#pragma unroll
    for (int i = 0; i < 3; i++) c += lam[i] * v[i][d];
    cb.c[d] = c;
  }
  auto dist2 = [&](const double *p) {
    double dd = 0;
#pragma unroll
    for (int d = 0; d < 3; d++) dd += (p[d] - cb.c[d]) * (p[d] - cb.c[d]);
    return dd;
  };
  double ds[4], r2 = dist2(bq);
#pragma unroll
  for (int s = 0; s < 4; s++) {
    ds[s] = dist2(sup[s]);
    if (lane & (1 << s)) r2 = fmax(r2, ds[s]);
  }
#pragma unroll
  for (int s = 0; s < 4; s++)
    if (s < ns && !(lane & (1 << s)) && ds[s] > r2 * (1 + 1e-12)) ok = false;
  cb.r2 = r2;
  return ok;
}

constexpr double kBallTol = 1e-13;

// Smallest ball over the points one block of NW waves can enumerate.
//   p0          point 0, where the iteration starts,
//   scan(b, f)  calls f(i, q) for this thread's share of the points, in any
//               order; points inside the ball b may be left out.
// Per iteration the point of largest excess is found with ties going to the
// lowest index (thread, wave, then block argmax), so the sequence of support
// sets -- and hence the ball -- does not depend on NW.  s_e / s_i hold 8 x NW
// and 2 x NW slots (double-buffered: one barrier per iteration).
//
// The top levels are a few blocks, whose time is the latency of one iteration
// after another.  So the reductions are register moves (DPP) instead of
// shuffles through the LDS unit, the point of largest excess travels with its
// excess instead of being looked up again, and the winning candidate's ball
// is read from the lane that solved it.  Plummer N = 2^20, p = 12: leaves 254
// -> 157 us, the twelve internal levels 1,000 -> 450 us, a top level 65 -> 29 us.
template <int NW, class Scan>
__device__ DBall block_minball(const double (&p0)[3], Scan scan, double *s_e, int *s_i) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = threadIdx.x / kWave;
  const BallLane mine = ball_lane(lane);
  DBall b;
  double sup[4][3];
  int ns = 1;
  for (int d = 0; d < 3; d++) b.c[d] = sup[0][d] = sup[1][d] = sup[2][d] = sup[3][d] = p0[d];
  b.r2 = 0;
  for (int iter = 0; iter < 10000; iter++) {
    double best = -1, bq[3] = {0, 0, 0};
    int bidx = 0x7fffffff;
    scan(b, [&](int i, const double *q) {
      double e = 0;
      for (int d = 0; d < 3; d++) e += (q[d] - b.c[d]) * (q[d] - b.c[d]);
      e -= b.r2;
      if (e > best || (e == best && i < bidx)) {
        best = e;
        bidx = i;
        for (int d = 0; d < 3; d++) bq[d] = q[d];
      }
    });
    // the wave's point: largest excess, ties to the lowest index
    const double wbest = wave_max(best);
    unsigned long long tied = __ballot(best == wbest);
    int src = __ffsll(tied) - 1, widx = __builtin_amdgcn_readlane(bidx, src);
    for (tied &= tied - 1; tied && wbest > 0; tied &= tied - 1) {
      const int l = __ffsll(tied) - 1, i = __builtin_amdgcn_readlane(bidx, l);
      if (i < widx) {
        widx = i;
        src = l;
      }
    }
    best = wbest;
    for (int d = 0; d < 3; d++) bq[d] = lane_value(bq[d], src);
    if (NW > 1) {
      const int par = iter & 1;
      double *se = s_e + par * 4 * NW;
      int *si = s_i + par * NW;
      if (lane == 0) {
        se[4 * wid] = best;
        for (int d = 0; d < 3; d++) se[4 * wid + 1 + d] = bq[d];
        si[wid] = widx;
      }
      __syncthreads();
      best = se[0];
      widx = si[0];
      int wb = 0;
      for (int w = 1; w < NW; w++) {
        const double e2 = se[4 * w];
        const int i2 = si[w];
        if (e2 > best || (e2 == best && i2 < widx)) {
          best = e2;
          widx = i2;
          wb = w;
        }
      }
      for (int d = 0; d < 3; d++) bq[d] = se[4 * wb + 1 + d];
    }
    if (best <= kBallTol * b.r2 || best <= 0) break;
    // the <= 15 candidates (subsets of the support) one per lane; the valid
    // one of smallest radius wins, ties to the lowest mask (the order a
    // sequential scan over masks would keep)
    DBall cb;
    const bool ok = candidate_ball(lane, mine, ns, bq, sup, cb);
    const double key = ok ? cb.r2 : INFINITY;
    const double kmin = row0_min(key);
    if (!(kmin < INFINITY)) break;  // numerically degenerate; keep the current ball
    const int bestmask = __ffsll(__ballot(key == kmin)) - 1;
    DBall bestb;
    for (int d = 0; d < 3; d++) bestb.c[d] = lane_value(cb.c[d], bestmask);
    bestb.r2 = kmin;
    // the new support: bq, then the chosen points in support order
    double nsup[4][3];
    int k = 1;
#pragma unroll
    for (int d = 0; d < 3; d++)
      nsup[0][d] = nsup[1][d] = nsup[2][d] = nsup[3][d] = bq[d];
#pragma unroll
    for (int s2 = 0; s2 < 4; s2++)
      if (bestmask & (1 << s2)) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
          nsup[1][d] = k == 1 ? sup[s2][d] : nsup[1][d];
          nsup[2][d] = k == 2 ? sup[s2][d] : nsup[2][d];
          nsup[3][d] = k == 3 ? sup[s2][d] : nsup[3][d];
        }
        k++;
      }
#pragma unroll
    for (int s2 = 0; s2 < 4; s2++)
#pragma unroll
      for (int d = 0; d < 3; d++) sup[s2][d] = nsup[s2][d];
    ns = k;
    const bool grew = bestb.r2 > b.r2;
    b = bestb;
    if (!grew) break;
  }
  return b;
}

// One wave, points 0..n-1 (n > 0) from get(), lane-strided scan.
template <class Get>
__device__ DBall wave_minball(int n, Get get) {
  const int lane = threadIdx.x & (kWave - 1);
  double p0[3];
  get(0, p0);
  return block_minball<1>(
      p0,
      [&](const DBall &, auto f) {
        for (int i = lane; i < n; i += kWave) {
          double q[3];
          get(i, q);
          f(i, q);
        }
      },
      nullptr, nullptr);
}

}  // namespace tcfmm
